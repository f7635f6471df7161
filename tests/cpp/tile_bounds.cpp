// Host-side check of the plain permutation tiles with 16-byte vectors at any element (kernels/perm_addr.hpp, the functions
// the kernel itself calls): every load and store of every thread of every workgroup lies inside its tensor and the LDS
// tile, and every element of B is written with the element of A that belongs there; workgroups are dealt to the dies
// without leaving a tile out.  Exit code 0 and "ok" on success.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../hiptensor_amd/csrc/host/permute_plan.hpp"
#include "../../hiptensor_amd/csrc/kernels/perm_addr.hpp"

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

struct Args // as the launcher fills its own
{
    uint32_t e_i, e_j, a_j, b_i, b_j, nt_i, nt_j, group;
    int32_t  nb;
    uint32_t bext[PERM_BATCH], ba[PERM_BATCH], bb[PERM_BATCH];
};

template <int W>
static void walk(const hiptk_permute_t& p, uint32_t TI, uint32_t TJ)
{
    Args a = {};
    const int mj = p.mode_j;
    a.e_i = (uint32_t)p.extent[0], a.e_j = (uint32_t)p.extent[mj], a.a_j = (uint32_t)p.a_stride[mj], a.b_i = (uint32_t)p.b_stride[0], a.b_j = 1;
    a.nt_i = (a.e_i + TI - 1) / TI, a.nt_j = (a.e_j + TJ - 1) / TJ;
    a.group       = p.group == 0 ? 0u : (uint32_t)p.group < a.nt_j ? (uint32_t)p.group : a.nt_j;
    uint32_t grid = a.nt_i * a.nt_j, n = 1;
    for(int d = 0; d < p.rank; d++)
        n *= (uint32_t)p.extent[d];
    for(int d = 1; d < p.rank; d++)
        if(d != mj)
        {
            a.bext[a.nb] = (uint32_t)p.extent[d], a.ba[a.nb] = (uint32_t)p.a_stride[d], a.bb[a.nb] = (uint32_t)p.b_stride[d];
            a.nb++;
            grid *= (uint32_t)p.extent[d];
        }
    // what B holds, by plain arithmetic
    std::vector<uint32_t> want(n), got(n, 0xFFFFFFFFu);
    for(uint32_t x = 0; x < n; x++)
    {
        uint32_t r = x, off = 0;
        for(int d = 0; d < p.rank; d++)
        {
            off += r % (uint32_t)p.extent[d] * (uint32_t)p.b_stride[d];
            r /= (uint32_t)p.extent[d];
        }
        want[off] = x;
    }
    for(int bands = 0; bands < 2; bands++)
    {
        std::vector<int> taken(grid, 0);
        std::fill(got.begin(), got.end(), 0xFFFFFFFFu);
        for(uint32_t b = 0; b < grid; b++)
        {
            const uint32_t work = tile_work(b, grid, bands != 0);
            CHECK(work < grid, "work %u of %u", work, grid);
            taken[work]++;
            uint32_t i0, j0, aoff, boff;
            tile_origin(a, work, TI, TJ, i0, j0, aoff, boff);
            CHECK(i0 < a.e_i && j0 < a.e_j, "tile %u at %u, %u", work, i0, j0);
            const uint32_t        nx = a.e_i - i0 < TI ? a.e_i - i0 : TI, ny = a.e_j - j0 < TJ ? a.e_j - j0 : TJ;
            std::vector<uint32_t> tile(TI * TJ, 0xFFFFFFFFu);
            if(nx >= W)
                for(uint32_t u = 0; u < TI / W * TJ; u++)
                {
                    const TileVector v = tile_vector<W, true>(u, TI / W, nx, ny);
                    if(!v.ok)
                        continue;
                    const uint32_t from = aoff + v.at + v.line * a.a_j;
                    CHECK(v.at + W <= nx && v.line < ny && from + W <= n, "load of %u elements at %u of %u", W, from, n);
                    for(uint32_t e = 0; e < W; e++)
                        tile[v.line * TI + v.at + e] = from + e;
                }
            else
                for(uint32_t u = 0; u < nx * ny; u++)
                    tile[u / nx * TI + u % nx] = aoff + u % nx + u / nx * a.a_j;
            if(ny >= W)
                for(uint32_t u = 0; u < TJ / W * TI; u++)
                {
                    const TileVector v = tile_vector<W, true>(u, TJ / W, ny, nx);
                    if(!v.ok)
                        continue;
                    const uint32_t to = boff + v.at + v.line * a.b_i;
                    CHECK(v.at + W <= ny && v.line < nx && to + W <= n, "store of %u elements at %u of %u", W, to, n);
                    for(uint32_t e = 0; e < W; e++)
                        got[to + e] = tile[(v.at + e) * TI + v.line];
                }
            else
                for(uint32_t u = 0; u < nx * ny; u++)
                    got[boff + u % ny + u / ny * a.b_i] = tile[u % ny * TI + u / ny];
        }
        for(uint32_t w = 0; w < grid; w++)
            CHECK(taken[w] == 1, "tile %u taken %d times of %u", w, taken[w], grid);
        for(uint32_t x = 0; x < n; x++)
            CHECK(got[x] == want[x], "B[%u] from %u, not %u", x, got[x], want[x]);
    }
}

int main()
{
    struct Case
    {
        std::vector<int64_t> len;
        std::vector<int>     perm;
    };
    const Case cases[] = {{{129, 150, 3}, {1, 0, 2}}, {{131, 5, 129}, {2, 1, 0}}, {{257, 259}, {1, 0}}, {{40, 300, 7}, {1, 2, 0}},
                          {{300, 41}, {1, 0}}, {{64, 3, 64, 2}, {2, 1, 0, 3}}, {{70, 2, 513}, {2, 0, 1}}, {{19, 25, 8}, {1, 0, 2}},
                          {{515, 33, 5}, {1, 2, 0}}, {{16, 1025}, {1, 0}}, {{3, 1027, 5}, {1, 2, 0}}, {{137, 9, 4, 265}, {3, 2, 1, 0}}};
    const uint32_t shapes4[4][2] = {{64, 64}, {256, 16}, {16, 256}, {128, 128}}, shapes2[4][2] = {{128, 128}, {512, 32}, {32, 512}, {256, 128}};
    int walked = 0;
    for(const Case& c : cases)
        for(int eb : {2, 4})
            for(int tile = 0; tile < 4; tile++)
                for(int group : {0, 1, 16})
                {
                    PermuteIn in;
                    in.elem_bytes = eb;
                    for(size_t d = 0; d < c.len.size(); d++)
                        in.lenA.push_back(c.len[d]), in.modeA.push_back((int)d), in.modeB.push_back(c.perm[d]), in.lenB.push_back(c.len[(size_t)c.perm[d]]);
                    in.A = (const void*)(uintptr_t)0x1002, in.B = (const void*)(uintptr_t)0x2004;
                    PermuteTuning t;
                    t.kernel = HIPTK_PERM_TILED, t.tile = tile, t.group = group, t.loose = true;
                    hiptk_permute_t p;
                    if(plan_permutation(in, t, p) != PermuteStatus::OK || p.kernel != HIPTK_PERM_TILED || !p.loose)
                    {
                        CHECK(false, "case of %zu modes not planned on loose tiles", c.len.size());
                        continue;
                    }
                    walked++;
                    if(eb == 4)
                        walk<4>(p, shapes4[p.tile][0], shapes4[p.tile][1]);
                    else
                        walk<8>(p, shapes2[p.tile][0], shapes2[p.tile][1]);
                }
    std::printf("%s: %d plans walked, %d failures\n", g_fail ? "FAILED" : "ok", walked, g_fail);
    return g_fail ? 1 : 0;
}
