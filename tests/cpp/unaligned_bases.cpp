// Host-side check of what runs where an operand's base is not aligned for the tile a plan chose: for problems planned by the
// library's planner, the register-staged tile the planner ranks best (not the class's largest), in its own number of slices.
// Exit code 0 and "ok" on success.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../hiptensor_amd/csrc/host/planner.hpp"
#include "../../hiptensor_amd/csrc/host/solution.hpp"
#include "../../include/hiptk_kernels.h"

using namespace hipta;

static int g_fail = 0;
#define CHECK(cond, ...)                                                   \
    do                                                                     \
    {                                                                      \
        if(!(cond))                                                        \
        {                                                                  \
            g_fail++;                                                      \
            std::printf("FAIL %s:%d %s: ", __FILE__, __LINE__, #cond);     \
            std::printf(__VA_ARGS__);                                      \
            std::printf("\n");                                             \
        }                                                                  \
    } while(0)

static TensorIn matrix(int dtype, int32_t fast, int64_t n, int32_t slow, int64_t m)
{
    TensorIn t;
    t.dtype = dtype, t.align = 16;
    t.mode = {fast, slow}, t.len = {n, m}, t.stride = {1, n};
    return t;
}

int main()
{
    struct Form
    {
        int     dtype, compute; // hipDataType, hiptensorComputeType_t
        int64_t m, n, k;
        int     off; // bytes the bases lie off a 16-byte boundary: less than the chosen tile takes
    };
    const Form forms[] = {
        {2, 4, 160, 768, 1152, 2}, {2, 4, 1024, 224, 800, 2}, {2, 4, 1600, 768, 2012, 2}, {2, 4, 2048, 512, 1480, 2},
        {2, 4, 256, 128, 102400, 2}, {2, 4, 8192, 16, 8192, 2}, {14, 4, 160, 768, 1152, 2}, {14, 4, 2048, 512, 1480, 2},
        {0, 4, 240, 120, 34560, 4}, {1, 16, 216, 120, 55680, 8}, {4, 2048, 256, 128, 65536, 8}, {5, 4096, 256, 256, 256, 8},
    };
    int walked = 0, sliced = 0;
    for(const Form& f : forms)
        for(int layout = 0; layout < 4; layout++)
        {
            ProblemIn in;
            in.A       = layout & 1 ? matrix(f.dtype, 20, f.k, 0, f.m) : matrix(f.dtype, 0, f.m, 20, f.k);
            in.B       = layout & 2 ? matrix(f.dtype, 20, f.k, 10, f.n) : matrix(f.dtype, 10, f.n, 20, f.k);
            in.D       = matrix(f.dtype, 0, f.m, 10, f.n);
            in.compute = f.compute;
            GemmView    v;
            std::string why;
            if(build_view(in, v, why) != PlanStatus::OK)
            {
                CHECK(false, "%s", why.c_str());
                continue;
            }
            std::vector<const Solution*> all = SolutionRegistry::get().forClass(v.cls);
            const auto                   ranked = rank_choices(all, v, 512ull << 20, DeviceModel());
            for(const Choice& c : ranked)
            {
                if(!c.sol->direct)
                    continue;
                char name[120];
                std::snprintf(name, sizeof(name), "class %d layout %d %lld x %lld x %lld tile %d in %d", v.cls, layout, (long long)v.P, (long long)v.Q,
                              (long long)v.K, c.sol->tile_id, c.split_k);
                CHECK(c.sol->vec_align == 4 || c.sol->vec_align == 16, "%s: bases of %d bytes", name, c.sol->vec_align);
                const Choice* o = stand_in(c, ranked);
                CHECK(o, "%s: nothing to stand in", name);
                if(!o)
                    continue;
                // the best staged choice there is, in the same slices where the tiles add in the same order
                const bool same_bits = v.cls != HIPTK_F16 && v.cls != HIPTK_BF16 && c.sol->bp == 64;
                CHECK(!same_bits || o->split_k == c.split_k, "%s: stand-in in %d", name, o->split_k);
                for(const Choice& s : ranked)
                    CHECK(s.sol->direct || (same_bits && s.split_k != c.split_k) || o->est_us <= s.est_us, "%s: %s in %d beats the stand-in", name, s.sol->name.c_str(), s.split_k);
                hiptk_problem_t p{};
                p.cls = v.cls, p.tile_id = c.sol->tile_id, p.split_k = c.split_k, p.P = v.P, p.Q = v.Q, p.K = v.K;
                p.x_kfast = v.x_kfast, p.y_kfast = v.y_kfast, p.x_vec = v.x_vec, p.y_vec = v.y_vec, p.k_affine = v.k_affine;
                p.shift_p = v.shift_p, p.shift_q = v.shift_q, p.xy_aligned = v.xy_aligned;
                p.x_max_off = (int32_t)v.x_max_off, p.y_max_off = (int32_t)v.y_max_off;
                p.unaligned_tile = o->sol->tile_id, p.unaligned_split = o->split_k;
                hiptk_problem_t want = p;
                want.tile_id         = o->sol->tile_id;
                for(int resolved = 0; resolved < 2; resolved++)
                {
                    if(resolved)
                        CHECK(hiptk_resolve(&p) == HIPTK_OK, "%s: resolve", name);
                    const std::string expect = hiptk_kernel_name(&want);
                    const void*       good   = (const void*)(uintptr_t)4096;
                    const void*       bad    = (const void*)(uintptr_t)(4096 + f.off);
                    CHECK(hiptk_kernel_name_at(&p, good, good) == std::string(hiptk_kernel_name(&p)), "%s: aligned", name);
                    if(f.off % c.sol->vec_align == 0)
                        continue;
                    CHECK(!expect.empty() && hiptk_kernel_name_at(&p, bad, good) == expect, "%s: X off: %s, not %s", name, hiptk_kernel_name_at(&p, bad, good),
                          expect.c_str());
                    CHECK(hiptk_kernel_name_at(&p, good, bad) == expect, "%s: Y off: %s, not %s", name, hiptk_kernel_name_at(&p, good, bad), expect.c_str());
                    walked++;
                    sliced += o->split_k > 1;
                }
            }
        }
    CHECK(walked >= 200 && sliced >= 50, "%d choices off their alignment, %d of them with slices", walked, sliced);

    // `xy_aligned` as a flag means 16 bytes
    hiptk_problem_t p{};
    p.cls = HIPTK_F16, p.tile_id = 11, p.x_kfast = p.y_kfast = 1, p.x_vec = p.y_vec = 8, p.k_affine = 1, p.P = p.Q = p.K = 512;
    p.x_max_off = p.y_max_off = 512 * 512 - 1;
    for(int a : {0, 1, 4, 16})
    {
        p.xy_aligned = a;
        CHECK(hiptk_kernel_available(&p) == (a == 1 || a == 16), "xy_aligned %d", a);
    }
    std::printf("%s: %d choices, %d failures\n", g_fail ? "FAILED" : "ok", walked, g_fail);
    return g_fail ? 1 : 0;
}
