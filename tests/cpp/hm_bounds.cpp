// Host-side check of the addressing of the 16-bit direct-load kernels with tiles of 64 and 128 rows (contract_hm.hpp, with the
// functions of hd_addr.hpp that the kernel itself calls): a direct load has no bounds check, so for random problems planned by
// the library's planner every request of every lane, K tile, split-K slice and (sampled) output tile is walked: it must read
// table entries inside the padded tables, start at a multiple of 4 bytes, lie inside the tensor, fetch the elements that the
// operand reads look for there, and every k of the problem must be multiplied once (the tile that K ends in: zeros beyond K).
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
    int64_t rstride() const { return v.cd_affine ? (is_x ? v.xp_stride : v.yq_stride) : 0; }
    int64_t kstride() const { return is_x ? v.xk_stride : v.yk_stride; }
    int64_t span() const { return (is_x != v.swapped) ? v.spanA : v.spanB; }
    int64_t row_offset(int r) const
    {
        CHECK((size_t)r < rtab().size(), "row table index %d of %zu", r, rtab().size());
        const int64_t off = rstride() ? (r < rows() ? r * rstride() : 0) : rtab()[(size_t)r];
        CHECK(r >= rows() || off == rtab()[(size_t)r], "computed row offset %lld, table %d", (long long)off, rtab()[(size_t)r]);
        return off;
    }
};

// the k that position `pos` of the tile at ko must hold (negative: zero): itself, or, where K ends inside a vector of eight
// k of a k-contiguous operand, the last eight k of K
static int64_t source_k(int64_t K, int ko, int pos, bool chunks)
{
    const int64_t first = ko + pos / 8 * 8;
    if(chunks && first < K && first + 8 > K)
        return K - 8 + pos % 8;
    return ko + pos < K ? ko + pos : -1;
}

template <bool KF, int BR>
static void walk_operand(const char* name, const Operand& o, int r0, const HmSlice& sl, bool chunks)
{
    constexpr int NL = BR / 32;
    const int64_t K  = o.v.K;
    for(int u = 0; u < sl.nt; u++)
    {
        const int  ko   = hm_origin(sl, u);
        const bool tail = u == 0 && sl.tail_k;
        CHECK(ko >= 0 && ko < K && (tail ? K - ko == sl.tail_k : ko + HK_BK <= K), "%s origin %d of K %lld", name, ko, (long long)K);
        std::vector<char> seen((size_t)BR * HK_BK, 0);
        for(int wave = 0; wave < 4; wave++)
            for(int i = 0; i < NL; i++)
                for(int lane = 0; lane < 64; lane++)
                {
                    const int     q    = (wave * NL + i) * 64 + lane;
                    const HdSlot  s    = hm_slot<KF, BR>(q);
                    const int     k    = tail ? hm_tail_k(s.k, sl.tail_k, chunks) : s.k;
                    const bool    zero = k == HM_ZERO;
                    const int64_t off  = o.row_offset(r0 + s.row) + (int64_t)(ko + k) * o.kstride();
                    g_walked++;
                    CHECK(s.row >= 0 && s.k >= 0 && s.row + (KF ? 1 : 8) <= BR && s.k + (KF ? 8 : 1) <= HK_BK, "%s slot -> row %d k %d", name, s.row, s.k);
                    for(int j = 0; j < 8; j++)
                    {
                        const int r = s.row + (KF ? 0 : j), pos = s.k + (KF ? j : 0);
                        // where the operand fetch looks for (r, pos)
                        const int want = KF ? r * HK_BK + 8 * hk_chunk_pos(r, pos / 8) + pos % 8 : pos * BR + hd_row_pos(r, pos);
                        CHECK(want == 8 * q + j, "%s (%d, %d) lands at %d, is read at %d", name, r, pos, 8 * q + j, want);
                        seen[(size_t)(r * HK_BK + pos)]++;
                        const int64_t source = source_k(K, ko, pos, chunks);
                        CHECK(zero == (source < 0), "%s k position %d of tile %d: zero %d", name, pos, ko, (int)zero);
                        if(!zero && r0 + r < o.rows())
                            CHECK(off + j == o.rtab()[(size_t)(r0 + r)] + source * o.kstride(), "%s (%d, %d) from %lld", name, r0 + r, ko + pos,
                                  (long long)(off + j));
                    }
                    if(!zero)
                    {
                        CHECK(off >= 0 && off + 8 <= o.span(), "%s elements %lld..+8 of %lld", name, (long long)off, (long long)o.span());
                        CHECK(off % 2 == 0, "%s element %lld is not at a multiple of 4 bytes", name, (long long)off);
                        CHECK(2ull * (uint64_t)(off + 8) <= 0xFFFFFFFFull - 3072, "%s offset beyond 32 bits", name);
                    }
                }
        for(char c : seen)
            CHECK(c == 1, "%s a stage element is filled %d times", name, (int)c);
        // a transposing read takes 4 rows at one k in one go
        for(int r = 0; !KF && r < BR; r += 4)
            for(int k = 0; k < 8; k++)
                CHECK(hd_row_pos(r + 3, k) == hd_row_pos(r, k) + 3 && hd_row_pos(r, k) % 4 == 0, "%s rows %d.. at k %d", name, r, k);
    }
}

template <int BP, int BQ>
static void walk(const char* name, const GemmView& v)
{
    const bool chunks = v.x_kfast || v.y_kfast;
    const int ktiles = (int)((v.K + HK_BK - 1) / HK_BK), tiles_p = (int)((v.P + BP - 1) / BP), tiles_q = (int)((v.Q + BQ - 1) / BQ);
    for(int want : {1, 2, 3, 5})
    {
        int split = std::min(want, ktiles);
        const int per = (ktiles + split - 1) / split;
        split         = (ktiles + per - 1) / per;
        std::vector<int> covered((size_t)v.K, 0);
        for(int z = 0; z < split; z++)
        {
            const HmSlice sl = hm_slice((int)v.K, z * per, per);
            CHECK(sl.nt >= 1, "%s empty slice", name);
            for(int u = 0; u < sl.nt; u++)
                for(int k = 0; k < HK_BK; k++)
                {
                    const int64_t s = source_k(v.K, hm_origin(sl, u), k, chunks);
                    // (as the kernel masks the operand registers of the first tile)
                    const int tk = u == 0 ? sl.tail_k : 0;
                    const bool masked = chunks && tk % 8 != 0 && k / 8 == tk / 8 && k % 8 < 8 - tk % 8;
                    if(s >= 0 && !masked)
                        covered[(size_t)s]++;
                }
            for(int corner = 0; corner < 4; corner++)
            {
                const int p_own = (corner & 1 ? tiles_p - 1 : 0) * BP, q_own = (corner & 2 ? tiles_q - 1 : 0) * BQ;
                const int p0 = (v.shift_p && p_own + BP > v.P) ? (int)v.P - BP : p_own;
                const int q0 = (v.shift_q && q_own + BQ > v.Q) ? (int)v.Q - BQ : q_own;
                CHECK(p0 >= 0 && q0 >= 0, "%s tile moved back beyond the start", name);
                if(v.x_kfast)
                    walk_operand<true, BP>(name, Operand{v, true}, p0, sl, chunks);
                else
                    walk_operand<false, BP>(name, Operand{v, true}, p0, sl, chunks);
                if(v.y_kfast)
                    walk_operand<true, BQ>(name, Operand{v, false}, q0, sl, chunks);
                else
                    walk_operand<false, BQ>(name, Operand{v, false}, q0, sl, chunks);
            }
        }
        for(int k = 0; k < v.K; k++)
            CHECK(covered[(size_t)k] == 1, "%s k %d multiplied %d times", name, k, covered[(size_t)k]);
    }
}

int main()
{
    std::mt19937 rng(5);
    auto         pick = [&](std::initializer_list<int> l) { return *(l.begin() + rng() % l.size()); };
    int          offered = 0, dword = 0, shifted = 0, tails = 0, plain = 0;
    for(int n = 0; n < 400; n++)
    {
        // modes 0 1 | 10 11 | 20 (21): rows, columns, reduction
        const int64_t m0 = pick({8, 16, 24, 33, 34, 62, 66, 70, 90, 128, 130}), m1 = pick({1, 1, 3, 4});
        const int64_t n0 = pick({8, 16, 40, 33, 50, 62, 66, 94, 128, 131}), n1 = pick({1, 1, 2, 5});
        const int64_t k0 = pick({64, 65, 66, 68, 72, 100, 126, 128, 130, 192, 250}), k1 = pick({1, 1, 2, 3});
        auto          tensor = [&](std::vector<std::pair<int, int64_t>> modes, int64_t pad) {
            TensorIn t;
            t.dtype   = 2;
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
        in.compute = 4;
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
        for(int tile = 13; tile <= 15; tile++)
        {
            hiptk_problem_t p{};
            p.cls = v.cls, p.tile_id = tile, p.x_kfast = v.x_kfast, p.y_kfast = v.y_kfast, p.x_vec = v.x_vec, p.y_vec = v.y_vec;
            p.k_affine = v.k_affine, p.P = v.P, p.Q = v.Q, p.K = v.K, p.shift_p = v.shift_p, p.shift_q = v.shift_q;
            p.xy_aligned = v.xy_aligned, p.x_max_off = (int32_t)v.x_max_off, p.y_max_off = (int32_t)v.y_max_off;
            if(!hiptk_kernel_available(&p))
                continue;
            offered++;
            (v.xy_aligned == 4 ? dword : plain)++;
            shifted += v.shift_p || v.shift_q;
            tails += v.K % 64 != 0;
            switch(tile)
            {
            case 13: walk<64, 64>(name, v); break;
            case 14: walk<128, 64>(name, v); break;
            default: walk<64, 128>(name, v); break;
            }
        }
    }
    CHECK(dword >= 100 && plain >= 50 && shifted >= 50 && tails >= 100, "offered %d: %d at 4 bytes, %d at 16, %d moved back, %d tails", offered, dword, plain,
          shifted, tails);
    std::printf("%s: %d (problem, tile) pairs (%d at 4 bytes, %d moved back, %d with a K tail), %ld requests, %d failures\n", g_fail ? "FAILED" : "ok", offered,
                dword, shifted, tails, g_walked, g_fail);
    return g_fail ? 1 : 0;
}
