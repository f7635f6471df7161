// Host-side check of the permutation kernels that move 16-byte vectors at any element (kernels/perm_addr.hpp, the
// functions the kernels themselves call): for a list of problems planned by the library's own planner this program walks
// every load and store of every thread and checks that it
//   * lies inside its tensor (and, for the grouped tiles, inside the LDS tile),
//   * takes from A what B holds there, and that every element of B is written.
// Exit code 0 and "ok" on success.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../hiptensor_amd/csrc/host/permute_plan.hpp"
#include "../../hiptensor_amd/csrc/kernels/perm_addr.hpp"

using namespace hipta;
using namespace hiptk;

static int g_fail = 0;
#define CHECK(cond, ...)                                                  \
    do                                                                    \
    {                                                                     \
        if(!(cond))                                                       \
        {                                                                 \
            if(g_fail < 20)                                               \
            {                                                             \
                std::printf("FAIL %s:%d %s: ", __FILE__, __LINE__, #cond); \
                std::printf(__VA_ARGS__);                                 \
                std::printf("\n");                                        \
            }                                                             \
            g_fail++;                                                     \
        }                                                                 \
    } while(0)

struct Case
{
    std::vector<int64_t> len;
    std::vector<int>     perm;
};

// element of A that B holds at every place, by plain arithmetic on the caller's lengths
static std::vector<uint32_t> sources(const Case& c)
{
    const size_t          r = c.len.size();
    std::vector<uint64_t> as(r);
    uint64_t              n = 1;
    for(size_t d = 0; d < r; d++)
    {
        as[d] = n;
        n *= (uint64_t)c.len[d];
    }
    std::vector<uint32_t> out((size_t)n);
    std::vector<int64_t>  at(r, 0);
    for(uint64_t b = 0; b < n; b++)
    {
        uint64_t a = 0;
        for(size_t k = 0; k < r; k++)
            a += (uint64_t)at[k] * as[(size_t)c.perm[k]];
        out[(size_t)b] = (uint32_t)a;
        for(size_t k = 0; k < r; k++)
        {
            if(++at[k] < c.len[(size_t)c.perm[k]])
                break;
            at[k] = 0;
        }
    }
    return out;
}

static void walk_runs(const hiptk_permute_t& p, const std::vector<uint32_t>& want)
{
    const uint32_t    n = (uint32_t)want.size(), V = 16u / (uint32_t)p.elem_bytes, last = n - V;
    const RunsShape   s = runs_shape(p, n);
    const uint32_t    U = (uint32_t)runs_per_thread(n, (int)V), per = PERM_THREADS * U * V;
    std::vector<char> written(n, 0);
    for(uint32_t blk = 0; blk < (n + per - 1) / per; blk++)
        for(uint32_t tid = 0; tid < (uint32_t)PERM_THREADS; tid++)
            for(uint32_t u = 0; u < U; u++)
            {
                const uint32_t   at = (blk * (PERM_THREADS * U) + tid) * V + u * PERM_THREADS * V, idx = at < last ? at : last;
                const RunsVector r = runs_vector(s, idx);
                CHECK((uint64_t)r.src + V <= n, "first load at %u of %u", r.src, n);
                CHECK(r.left >= V || (r.next >= r.left && (uint64_t)r.next - r.left + V <= n), "second load at %u - %u of %u", r.next, r.left, n);
                for(uint32_t e = 0; e < V; e++)
                {
                    const uint32_t from = e < r.left ? r.src + e : r.next - r.left + e;
                    CHECK(from == want[idx + e], "element %u of B from %u, not %u", idx + e, from, want[idx + e]);
                }
                if(at < n)
                    for(uint32_t e = 0; e < V; e++)
                        written[idx + e] = 1;
            }
    for(uint32_t b = 0; b < n; b++)
        CHECK(written[b], "element %u of %u is not written", b, n);
}

template <int V>
static void walk_group(const hiptk_permute_t& p, const std::vector<uint32_t>& want)
{
    const uint32_t        n    = (uint32_t)want.size();
    int64_t               grid = 0;
    const GroupShape      s    = group_shape(p, grid);
    const uint32_t        RV = group_per_line(s.w_i * s.c_i, V, true), CV = group_per_line(s.w_j * s.c_j, V, true);
    const size_t          lds = (size_t)s.w_j * s.c_j * s.pitch;
    std::vector<uint32_t> tile(lds);
    std::vector<char>     written(n, 0);
    for(int64_t blk = 0; blk < grid; blk++)
    {
        const GroupTile t = group_tile(s, (uint32_t)blk);
        tile.assign(lds, 0xFFFFFFFFu);
        auto read = [&](const GroupVector& g, uint32_t W) {
            const uint64_t from = (uint64_t)t.aoff + (g.ok ? g.at + g.off : 0u);
            CHECK(from + W <= n, "load of %u at %llu of %u", W, (unsigned long long)from, n);
            for(uint32_t e = 0; g.ok && e < W; e++)
            {
                const size_t at = (size_t)g.line * s.pitch + g.at + e;
                CHECK(at < lds, "LDS %zu of %zu", at, lds);
                if(at < lds)
                    tile[at] = (uint32_t)from + e;
            }
        };
        auto write = [&](const GroupVector& g, uint32_t W) {
            const uint64_t to = (uint64_t)t.boff + g.at + g.off;
            CHECK(!g.ok || to + W <= n, "store of %u at %llu of %u", W, (unsigned long long)to, n);
            for(uint32_t e = 0; g.ok && to + W <= n && e < W; e++)
            {
                const size_t at = (size_t)(g.at + e) * s.pitch + g.line;
                CHECK(at < lds && tile[at] == want[(size_t)to + e], "element %llu of B", (unsigned long long)to + e);
                written[(size_t)to + e] = 1;
            }
        };
        // (all threads of all passes: whole rounds of eight vectors a thread when reading)
        const uint32_t round = PERM_THREADS * 8, rs = group_singles(t.nx), ws = group_singles(t.ny);
        if(t.nx >= (uint32_t)V)
            for(uint32_t v = 0; v < (RV * t.ny + round - 1) / round * round; v++)
                read(group_read<V, true>(s, t, v, RV, s.m_rv), V);
        else
            for(uint32_t v = 0; v < (rs * t.ny + round - 1) / round * round; v++)
                read(group_read<1, true>(s, t, v, rs, recip(rs)), 1);
        if(t.ny >= (uint32_t)V)
            for(uint32_t v = 0; v < CV * t.nx; v++)
                write(group_write<V, true>(s, t, v, CV, s.m_cv), V);
        else
            for(uint32_t v = 0; v < ws * t.nx; v++)
                write(group_write<1, true>(s, t, v, ws, recip(ws)), 1);
    }
    for(uint32_t b = 0; b < n; b++)
        CHECK(written[b], "element %u of %u is not written", b, n);
}

int main()
{
    // runs of exactly a vector and little more, long odd ones, one vector and four per thread;
    // tiles whose last row or column is shorter than a vector (down to one element) or a little longer, chunks that do
    // not divide their modes
    const Case cases[] = {
        {{4, 2, 3}, {0, 2, 1}},
        {{8, 3, 2}, {0, 2, 1}},
        {{9, 2, 2}, {0, 2, 1}},
        {{11, 7, 5}, {0, 2, 1}},
        {{15, 2, 3, 4}, {0, 3, 2, 1}},
        {{17, 3, 5, 2, 4}, {0, 4, 2, 3, 1}},
        {{30, 7, 11, 7, 3, 5}, {0, 4, 2, 3, 1, 5}},
        {{41, 61, 13}, {0, 2, 1}},
        {{229, 6, 5, 7}, {0, 3, 2, 1}},
        {{1659, 20, 3, 2}, {0, 2, 3, 1}},
        {{4099, 2, 3}, {0, 2, 1}},
        {{63, 256, 261}, {0, 2, 1}},
        {{127, 256, 259}, {0, 2, 1}},
        {{129, 150, 131}, {2, 1, 0}},
        {{131, 129, 200}, {1, 0, 2}},
        {{137, 171, 129}, {2, 1, 0}},
        {{67, 305, 129}, {2, 1, 0}},
        {{21, 25, 23, 31, 25}, {4, 2, 1, 3, 0}},
        {{19, 7, 49, 9, 57}, {3, 4, 2, 1, 0}},
        {{65, 513, 129}, {1, 2, 0}},
        {{13, 11, 7, 9, 15, 35}, {4, 2, 3, 0, 5, 1}},
    };
    int runs = 0, groups = 0;
    for(const Case& c : cases)
        for(int eb : {2, 4})
        {
            PermuteIn in;
            in.elem_bytes = eb;
            in.lenA       = c.len;
            for(size_t d = 0; d < c.len.size(); d++)
            {
                in.modeA.push_back((int32_t)d);
                in.modeB.push_back(c.perm[d]);
                in.lenB.push_back(c.len[(size_t)c.perm[d]]);
            }
            in.A = in.B = reinterpret_cast<const void*>((uintptr_t)256);
            PermuteTuning tune;
            tune.kernel       = c.perm[0] == 0 ? HIPTK_PERM_RUNS : HIPTK_PERM_GROUPED;
            hiptk_permute_t p = {};
            CHECK(plan_permutation(in, tune, p) == PermuteStatus::OK, "plan");
            const std::vector<uint32_t> want = sources(c);
            if(p.kernel == HIPTK_PERM_RUNS)
            {
                walk_runs(p, want);
                runs++;
            }
            else if(p.kernel == HIPTK_PERM_GROUPED && p.loose)
            {
                eb == 4 ? walk_group<4>(p, want) : walk_group<8>(p, want);
                groups++;
            }
        }
    // division by reciprocals: exact for every 32-bit index, at the multiples where it could slip
    for(uint32_t e : {2u, 3u, 5u, 7u, 64u, 127u, 229u, 641u, 1659u, 4096u, 65537u, 6700417u, 1073741823u})
        for(uint64_t q = 0; q * e <= 0x7FFFFFFFull; q += 1 + q / 1024)
            for(int64_t x = (int64_t)(q * e) - 1; x <= (int64_t)(q * e) + 1; x++)
            {
                uint32_t rem = 0;
                if(x >= 0 && x <= 0x7FFFFFFFll)
                    CHECK(div_by((uint32_t)x, e, magic_of(e), rem) == (uint32_t)x / e && rem == (uint32_t)x % e, "%lld / %u", (long long)x, e);
            }
    CHECK(runs == 25 && groups == 16, "%d linear problems, %d of loose tiles", runs, groups);
    std::printf(g_fail ? "%d failures\n" : "ok\n", g_fail);
    return g_fail ? 1 : 0;
}
