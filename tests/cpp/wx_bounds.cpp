// Host-side check of the addressing of the 32/64-bit direct-load kernels that take operands at any element (contract_wx_kernel in
// contract_wd.hpp, with the functions of hd_addr.hpp that the kernel itself calls): a direct load has no bounds check, so for
// random problems planned by the library's planner every request of every lane, K tile, split-K slice and wave that splits K is
// walked, for the corner tiles: it must read table entries inside the padded tables, lie inside the tensor and fetch the elements
// that the operand reads look for, and every k must be multiplied once (the tile that K ends in: zeros beyond K).
// Exit code 0 and "ok" on success.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../../hiptensor_amd/csrc/host/planner.hpp"
#include "../../hiptensor_amd/csrc/kernels/hd_addr.hpp"
#include "../../include/hiptk_kernels.h"

using namespace hipta;
using namespace hiptk;

static int g_fail = 0;
#define CHECK(cond, ...)                                                   \
    do                                                                     \
    {                                                                      \
        if(!(cond))                                                        \
        {                                                                  \
            if(g_fail++ < 20)                                              \
            {                                                              \
                std::printf("FAIL %s:%d %s: ", __FILE__, __LINE__, #cond); \
                std::printf(__VA_ARGS__);                                  \
                std::printf("\n");                                         \
            }                                                              \
        }                                                                  \
    } while(0)

static long g_walked = 0;

// the element offset of (row, k) of an operand as the kernel computes it
struct Operand
{
    const GemmView& v;
    bool            is_x;
    const std::vector<int32_t>& rtab() const { return is_x ? v.xp : v.yq; }
    int64_t rows() const { return is_x ? v.P : v.Q; }
    // (these kernels read the row tables)
    int64_t row_offset(int r) const
    {
        CHECK((size_t)r < rtab().size(), "row table index %d of %zu", r, rtab().size());
        return rtab()[(size_t)r];
    }
    int64_t kstride() const { return is_x ? v.xk_stride : v.yk_stride; }
    int64_t span() const { return (is_x != v.swapped) ? v.spanA : v.spanB; }
};

// the k that position `pos` of the tile at ko must hold (negative: zero)
template <int V>
static int64_t source_k(int64_t K, int ko, int pos, bool chunks)
{
    const int64_t first = ko + pos / V * V;
    if(chunks && first < K && first + V > K)
        return K - V + pos % V;
    return ko + pos < K ? ko + pos : -1;
}

// one K tile of an operand: `tail` > 0: the short last one
template <int V, int BK, bool KF, int ROWS>
static void walk_tile(const char* name, const Operand& o, int r0, int ko, int tail, bool chunks)
{
    std::vector<char> seen((size_t)ROWS * BK, 0);
    for(int q = 0; q < ROWS * BK / V; q++)
    {
        const HdSlot  s    = KF ? wd_slot_kf<V, ROWS>(q) : wd_slot<V, ROWS>(q);
        const int     k    = tail ? wd_short_k<V>(s.k, tail, chunks) : s.k;
        const bool    zero = k == WD_ZERO;
        const int64_t off  = o.row_offset(r0 + s.row) + (int64_t)(ko + k) * o.kstride();
        g_walked++;
        for(int j = 0; j < V; j++)
        {
            const int r = s.row + (KF ? 0 : j), pos = s.k + (KF ? j : 0);
            const int want = KF ? (pos / V * ROWS + r) * V + pos % V : pos * ROWS + r;
            CHECK(want == V * q + j, "%s (%d, %d) lands at %d, is read at %d", name, r, pos, V * q + j, want);
            seen[(size_t)(r * BK + pos)]++;
            const int64_t source = source_k<V>(o.v.K, ko, pos, chunks);
            CHECK(zero == (source < 0), "%s k position %d of tile %d: zero %d", name, pos, ko, (int)zero);
            if(!zero && r0 + r < o.rows())
                CHECK(off + j == o.rtab()[(size_t)(r0 + r)] + source * o.kstride(), "%s (%d, %d) from %lld", name, r0 + r, ko + pos, (long long)(off + j));
        }
        if(!zero)
            CHECK(ko + k >= 0 && off >= 0 && off + V <= o.span(), "%s elements %lld..+%d of %lld", name, (long long)off, V, (long long)o.span());
    }
    for(char c : seen)
        CHECK(c == 1, "%s a stage element is filled %d times", name, (int)c);
}

template <int V, int BK, int ROWS, bool WK>
static void walk(const char* name, const GemmView& v)
{
    const bool chunks = v.x_kfast || v.y_kfast;
    const int  K = (int)v.K, ktiles = (K + BK - 1) / BK, tiles_p = (int)((v.P + ROWS - 1) / ROWS), tiles_q = (int)((v.Q + ROWS - 1) / ROWS);
    for(int want : {1, 2, 3, 5})
    {
        int       split = std::min(want, ktiles);
        const int per   = (ktiles + split - 1) / split;
        split           = (ktiles + per - 1) / per;
        std::vector<int> covered((size_t)K, 0);
        for(int z = 0; z < split; z++)
            for(int w = 0; w < (WK ? 4 : 1); w++)
            {
                int begin = z * per, end = std::min(begin + per, ktiles);
                if(WK)
                {
                    const WdChunk c = wd_wave_chunk(end - begin, w);
                    begin += c.first, end = begin + c.count;
                }
                const int nt = end - begin;
                if(nt <= 0)
                    continue;
                // (as the kernel orders them: the short last tile first, then the whole ones; requests beyond the last repeat it)
                const int short_k = end == ktiles ? K % BK : 0;
                const int klast   = short_k ? (nt > 1 ? (begin + nt - 2) * BK : 0) : (begin + nt - 1) * BK;
                int       ko      = short_k && nt == 1 ? 0 : begin * BK;
                for(int u = 0; u < nt + 4; u++)
                {
                    const bool first = short_k && u == 0, real = u < nt;
                    const int  at    = first ? (ktiles - 1) * BK : ko;
                    CHECK(at >= 0 && (first || at + BK <= K), "%s tile at %d of K %d", name, at, K);
                    for(int k = 0; real && k < BK; k++)
                    {
                        const int64_t s    = source_k<V>(K, at, k, chunks);
                        const bool masked = first && chunks && short_k % V != 0 && k / V == short_k / V && k % V < V - short_k % V;
                        if(s >= 0 && !masked)
                            covered[(size_t)s]++;
                    }
                    for(int corner = 0; corner < 4; corner++)
                    {
                        const int p_own = (corner & 1 ? tiles_p - 1 : 0) * ROWS, q_own = (corner & 2 ? tiles_q - 1 : 0) * ROWS;
                        const int p0 = v.shift_p && p_own + ROWS > v.P ? (int)v.P - ROWS : p_own;
                        const int q0 = v.shift_q && q_own + ROWS > v.Q ? (int)v.Q - ROWS : q_own;
                        CHECK(p0 >= 0 && q0 >= 0, "%s tile moved back beyond the start", name);
                        const Operand x{v, true}, y{v, false};
                        v.x_kfast ? walk_tile<V, BK, true, ROWS>(name, x, p0, at, first ? short_k : 0, chunks)
                                  : walk_tile<V, BK, false, ROWS>(name, x, p0, at, first ? short_k : 0, chunks);
                        v.y_kfast ? walk_tile<V, BK, true, ROWS>(name, y, q0, at, first ? short_k : 0, chunks)
                                  : walk_tile<V, BK, false, ROWS>(name, y, q0, at, first ? short_k : 0, chunks);
                    }
                    if(!first)
                        ko = wd_next_origin(ko, klast, BK);
                }
            }
        for(int k = 0; k < K; k++)
            CHECK(covered[(size_t)k] == 1, "%s k %d multiplied %d times", name, k, covered[(size_t)k]);
    }
}

int main()
{
    std::mt19937 rng(5);
    auto         pick = [&](std::initializer_list<int> l) { return *(l.begin() + rng() % l.size()); };
    int          offered = 0, dword = 0, shifted = 0, tails = 0, inside = 0;
    for(int n = 0; n < 400; n++)
    {
        // modes 0 1 | 10 11 | 20 (21): rows, columns, reduction
        const int64_t m0 = pick({8, 16, 24, 33, 34, 62, 66, 70, 90, 128, 130}), m1 = pick({1, 1, 3, 4});
        const int64_t n0 = pick({8, 16, 40, 33, 50, 62, 66, 94, 128, 131}), n1 = pick({1, 1, 2, 5});
        const int64_t k0 = pick({8, 9, 16, 17, 18, 21, 23, 32, 33, 50, 63}), k1 = pick({1, 1, 2, 3});
        const int     cls = n % 3; // f32, f64, complex f32
        auto          tensor = [&](std::vector<std::pair<int, int64_t>> modes, int64_t pad) {
            TensorIn t;
            t.dtype   = cls == 0 ? 0 : cls == 1 ? 1 : 4;
            t.align   = 256;
            int64_t s = 1;
            for(size_t i = 0; i < modes.size(); i++)
            {
                t.mode.push_back(modes[i].first), t.len.push_back(modes[i].second), t.stride.push_back(s);
                s = s * modes[i].second + (i == 0 ? pad : 0);
            }
            return t;
        };
        std::vector<std::pair<int, int64_t>> M{{0, m0}, {1, m1}}, N{{10, n0}, {11, n1}}, K{{20, k0}, {21, k1}};
        auto cat = [](std::vector<std::pair<int, int64_t>> a, const std::vector<std::pair<int, int64_t>>& b) {
            a.insert(a.end(), b.begin(), b.end());
            return a;
        };
        ProblemIn in;
        const int form = (int)(rng() % 4);
        const int64_t pad = k1 == 1 ? pick({0, 0, 1, 2}) : 0; // (a padded leading dimension: k may be odd where it is contiguous)
        in.A = tensor(form & 1 ? cat(M, K) : cat(K, M), pad);
        in.B = tensor(form & 2 ? cat(N, K) : cat(K, N), pad);
        in.D = tensor(cat(M, N), 0);
        in.bilinear = rng() % 2 != 0;
        if(in.bilinear)
            in.C = in.D;
        in.compute = cls == 0 ? 4 : cls == 1 ? 16 : 2048;
        GemmView    v;
        std::string why;
        if(build_view(in, v, why) != PlanStatus::OK)
        {
            CHECK(false, "%s", why.c_str());
            continue;
        }
        char name[160];
        std::snprintf(name, sizeof(name), "P %lld Q %lld K %lld kf %d%d shift %d%d pad %lld", (long long)v.P, (long long)v.Q, (long long)v.K, v.x_kfast,
                      v.y_kfast, v.shift_p, v.shift_q, (long long)pad);
        for(int tile = 4; tile <= 5; tile++)
        {
            hiptk_problem_t p{};
            p.cls = v.cls, p.tile_id = tile, p.x_kfast = v.x_kfast, p.y_kfast = v.y_kfast, p.x_vec = v.x_vec, p.y_vec = v.y_vec;
            p.k_affine = v.k_affine, p.P = v.P, p.Q = v.Q, p.K = v.K, p.shift_p = v.shift_p, p.shift_q = v.shift_q;
            p.xy_aligned = v.xy_aligned, p.x_max_off = (int32_t)v.x_max_off, p.y_max_off = (int32_t)v.y_max_off;
            if(!hiptk_kernel_available(&p))
                continue;
            offered++;
            dword += v.xy_aligned == 4;
            shifted += v.shift_p || v.shift_q;
            tails += v.K % (cls == 0 ? 16 : 8) != 0;
            inside += (v.x_kfast || v.y_kfast) && v.K % (cls == 0 ? 4 : 2) != 0;
            if(cls == 0)
                tile == 4 ? walk<4, 16, 64, false>(name, v) : walk<4, 16, 32, true>(name, v);
            else
                tile == 4 ? walk<2, 8, 64, false>(name, v) : walk<2, 8, 32, true>(name, v);
        }
    }
    CHECK(dword >= 50 && shifted >= 50 && tails >= 100 && inside >= 20, "offered %d: %d at 4 bytes, %d moved back, %d tails, %d inside a vector", offered, dword,
          shifted, tails, inside);
    std::printf("%s: %d (problem, tile) pairs (%d at 4 bytes, %d moved back, %d with a K tail, %d of them inside a vector), %ld requests, %d failures\n",
                g_fail ? "FAILED" : "ok", offered, dword, shifted, tails, inside, g_walked, g_fail);
    return g_fail ? 1 : 0;
}
