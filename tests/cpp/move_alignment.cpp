// Host-side check of the alignment a planned move asks of its source: a source at a multiple of 16 bytes whose layout admits
// vectors there is refused below their alignment by every kernel that was chosen where one that reads such vectors would be
// allowed, also by those that could read it at any element.  Exit code 0 and "ok" on success.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../hiptensor_amd/csrc/host/permute_plan.hpp"

using namespace hipta;

static int g_fail = 0;

// bytes that A must start at a multiple of for hiptk_permute to take `p`
static int needs(const hiptk_permute_t& p)
{
    const int by_vec = p.kernel == HIPTK_PERM_GATHER || p.kernel == HIPTK_PERM_RUNS || p.loose ? p.elem_bytes : p.vec_r * p.elem_bytes;
    return p.a_align > by_vec ? p.a_align : by_vec;
}

int main()
{
    struct Form
    {
        int                  elem_bytes;
        std::vector<int64_t> len;
        std::vector<int>     perm; // mode k of B is mode perm[k] of A
        int                  kernel, loose, bytes;
    };
    const Form forms[] = {
        {2, {3000, 2057}, {1, 0}, HIPTK_PERM_GROUPED, 1, 16}, // single elements on B's side, up to 2^23
        {2, {8000, 4101}, {1, 0}, HIPTK_PERM_TILED, 1, 16}, // ... and beyond
        {2, {8002, 4101}, {1, 0}, HIPTK_PERM_TILED, 1, 4},
        {2, {8001, 4101}, {1, 0}, HIPTK_PERM_TILED, 1, 2},
        {4, {2002, 4101}, {1, 0}, HIPTK_PERM_TILED, 1, 8}, // f32 read in less than 16 bytes
        {4, {2004, 4101}, {1, 0}, HIPTK_PERM_TILED, 0, 16},
        {2, {16, 24, 48, 40, 32}, {1, 0, 2, 4, 3}, HIPTK_PERM_GATHER, 0, 16}, // blocks transposed in place
        {4, {20, 24, 230, 28}, {1, 0, 3, 2}, HIPTK_PERM_GATHER, 0, 16},
        {4, {60000, 57}, {1, 0}, HIPTK_PERM_TILED, 0, 16}, // strips of a small tensor
        {2, {56, 52296}, {1, 0}, HIPTK_PERM_GROUPED, 0, 16},
        {2, {120, 128}, {1, 0}, HIPTK_PERM_GATHER, 0, 2}, // up to 16384 elements: any, as ever
    };
    for(const Form& f : forms)
        for(int align : {16, f.elem_bytes})
        {
            PermuteIn in;
            in.elem_bytes = f.elem_bytes;
            in.lenA       = f.len;
            for(size_t i = 0; i < f.len.size(); i++)
            {
                in.modeA.push_back((int32_t)i);
                in.modeB.push_back(f.perm[i]);
                in.lenB.push_back(f.len[(size_t)f.perm[i]]);
            }
            in.A = reinterpret_cast<const void*>((uintptr_t)align);
            in.B = reinterpret_cast<const void*>((uintptr_t)256);
            PermuteTuning tune;
            tune.gather = false; // as the moves into packed copies are planned
            hiptk_permute_t p{};
            const int       bytes = align == 16 ? f.bytes : f.elem_bytes;
            if(plan_permutation(in, tune, p) != PermuteStatus::OK || (align == 16 && (p.kernel != f.kernel || p.loose != f.loose)) || needs(p) != bytes)
            {
                g_fail++;
                std::printf("FAIL %d bytes %lld x %lld ... source at %d: kernel %d loose %d asks %d, not %d\n", f.elem_bytes, (long long)f.len[0],
                            (long long)f.len[1], align, p.kernel, p.loose, needs(p), bytes);
            }
        }
    std::printf("%s: %d failures\n", g_fail ? "FAILED" : "ok", g_fail);
    return g_fail ? 1 : 0;
}
