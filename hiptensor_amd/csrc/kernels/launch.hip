// Kernel-layer C ABI: kernel registry lookup, argument checks, launch, and the
// split-K reduction kernels.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "contract_h.hpp"
#include "contract_w.hpp"
#include "dma_lds.hpp"

namespace hiptk
{
    namespace
    {
        struct Registry
        {
            std::vector<KernelEntry> all;
            Registry()
            {
                typedef const KernelEntry* (*src_fn)(int*);
                const src_fn sources[] = {entries_f16_hd,
                                          entries_f16_hd192,
                                          entries_f16_hd192_tab,
                                          entries_bf16_hd,
                                          entries_bf16_hd192,
                                          entries_bf16_hd192_tab,
                                          entries_f16_hk_kx,
                                          entries_f16_hk_rx,
                                          entries_bf16_hk_kx,
                                          entries_bf16_hk_rx,
                                          entries_f16_hr192_kx,
                                          entries_f16_hr192_rx,
                                          entries_bf16_hr192_kx,
                                          entries_bf16_hr192_rx,
                                          entries_f16_hm,
                                          entries_bf16_hm,
                                          entries_f16_aff,
                                          entries_bf16_aff,
                                          entries_f16_vec,
                                          entries_f16_gen,
                                          entries_bf16_vec,
                                          entries_bf16_gen,
                                          entries_f16_v4,
                                          entries_f16_v2,
                                          entries_bf16_v4,
                                          entries_bf16_v2,
                                          entries_f32,
                                          entries_f64,
                                          entries_f32_any,
                                          entries_f64_any,
                                          entries_c32_any,
                                          entries_c32,
                                          entries_c64,
                                          entries_f64_as_f32,
                                          entries_f32_as_f16,
                                          entries_f32_as_bf16};
                for(src_fn f : sources)
                {
                    int                n = 0;
                    const KernelEntry* e = f(&n);
                    all.insert(all.end(), e, e + n);
                }
            }
        };

        const Registry& registry()
        {
            static const Registry r;
            return r;
        }

        int acc_bytes(int cls)
        {
            switch(cls)
            {
            case HIPTK_F64: return 8;
            case HIPTK_C32: return 8;
            case HIPTK_C64: return 16;
            default: return 4;
            }
        }

        // bytes of one operand element in memory
        int operand_bytes(int cls)
        {
            switch(cls)
            {
            case HIPTK_F16:
            case HIPTK_BF16: return 2;
            case HIPTK_F64:
            case HIPTK_F64_AS_F32:
            case HIPTK_C32: return 8;
            case HIPTK_C64: return 16;
            default: return 4;
            }
        }

        // ---- split-K reduction: sum the partials in slice order, apply alpha / beta ----

        struct FinF16
        {
            typedef float    O;
            typedef uint16_t E;
            static __device__ inline E finish(O x, const double* al, const double* be, bool bil, const E* c)
            {
                float v = (float)al[0] * x;
                if(bil)
                    v += (float)be[0] * TraitsF16::to_f32(*c);
                return TraitsF16::from_f32(v);
            }
            static __device__ inline O add(O a, O b) { return a + b; }
        };

        struct FinBF16
        {
            typedef float    O;
            typedef uint16_t E;
            static __device__ inline E finish(O x, const double* al, const double* be, bool bil, const E* c)
            {
                float v = (float)al[0] * x;
                if(bil)
                    v += (float)be[0] * TraitsBF16::to_f32(*c);
                return TraitsBF16::from_f32(v);
            }
            static __device__ inline O add(O a, O b) { return a + b; }
        };

        template <typename Tr>
        struct FinWide
        {
            typedef typename Tr::O O;
            typedef typename Tr::E E;
            static __device__ inline E finish(O x, const double* al, const double* be, bool bil, const E* c)
            {
                return Tr::finish(x, al, be, bil, c);
            }
            static __device__ inline float   add(float a, float b) { return a + b; }
            static __device__ inline double  add(double a, double b) { return a + b; }
            static __device__ inline float2  add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
            static __device__ inline double2 add(double2 a, double2 b)
            {
                return make_double2(a.x + b.x, a.y + b.y);
            }
        };

        // Sum of the split-K partials, and the epilogue.  Bound by the latency of its loads where outputs are few, by the
        // caches and HBM where they are many.  A thread owns V consecutive outputs, has DEPTH slices' loads of them in
        // flight, takes what is left of its slices in fours, twos and ones (loads repeated to fill a batch cost 0.4 us at two
        // slices of few outputs and up to 1.2 of many), and looks up where the outputs go beside the loads.  DEALT: where
        // outputs leave the device idle the slices are dealt to 2^(8 - lane_bits) threads of the workgroup, `per`
        // consecutive ones each, whose sums are added up through LDS in slice order.  One thread per output that walks
        // the slices one load after another takes 4-5 us for 8 slices, 9.5 for 32 and 16-20 for 64, whatever the
        // size of the output; here f32 64 x 64 in 64 slices 3.3 (18.4), 90 x 80 in 32 2.9 (9.5), 256 x 256 in 32 3.4 (9.5), in 2
        // 2.5 (2.4), 1450 x 1450 in 4 7.3 (10.4), 2048 x 2048 in 2 9.1 (11.3).  Behind it: 16 and more slices of outputs of
        // 8 or 16 bytes that lie a power of two apart (c32 1024 x 1024 in 16 23.0 and 20.6; the planner cuts no such
        // output into so many).
        // The order of the sum depends on the problem alone: results are the same on every run.
        template <typename Fin, int V, bool DEALT, int DEPTH>
        __global__ void __launch_bounds__(256) splitk_reduce_kernel(const KArgs a, int lane_bits, int per)
        {
            static_assert(V == 1 || !DEALT, "dealt slices: one output a thread");
            typedef typename Fin::O O;
            typedef typename Fin::E E;
            struct Vec
            {
                O v[V];
            };
            struct Elems
            {
                E v[V];
            };
            const size_t total = (size_t)a.P * (size_t)a.Q;
            const int    lane  = DEALT ? (int)threadIdx.x & ((1 << lane_bits) - 1) : (int)threadIdx.x;
            const int    g     = DEALT ? (int)threadIdx.x >> lane_bits : 0;
            const size_t idx   = (((size_t)blockIdx.x << (DEALT ? lane_bits : 8)) + lane) * V;
            const bool   in    = idx < total;
            if(!DEALT && !in)
                return;
            // the last vector starts inside the tensor and may reach beyond it: it is loaded V elements from the end
            // of the slice (which holds more than V), and only its own outputs are kept
            const int  over = V > 1 && idx + V > total ? (int)(idx + V - total) : 0;
            const int  z0   = DEALT ? g * per : 0;
            const int  n    = !DEALT ? a.split_k : !in ? 0 : z0 + per < a.split_k ? per : a.split_k - z0;
            const bool bil  = a.bilinear != 0;
            // where the outputs go, and their elements of C: looked up beside the partials, not behind them
            // (an output vector may run over the end of a row of D)
            int p, q;
            if(total <= 0xFFFFFFFFull)
            {
                p = (int)((uint32_t)idx / (uint32_t)a.Q);
                q = (int)((uint32_t)idx % (uint32_t)a.Q);
            }
            else
            {
                p = (int)(idx / (size_t)a.Q);
                q = (int)(idx % (size_t)a.Q);
            }
            uint32_t doff[V], coff[V];
            bool     d_run = idx + V <= total, c_run = d_run; // one run of V elements of D / C
            Elems    c     = {};
#pragma unroll
            for(int e = 0; e < V; e++)
            {
                const bool ok = in && g == 0 && idx + e < total;
                const int  pe = ok ? p : 0, qe = ok ? q : 0;
                if(a.cd_affine)
                {
                    doff[e] = (uint32_t)pe * (uint32_t)a.dp_stride + (uint32_t)qe * (uint32_t)a.dq_stride;
                    coff[e] = (uint32_t)pe * (uint32_t)a.cp_stride + (uint32_t)qe * (uint32_t)a.cq_stride;
                }
                else
                {
                    doff[e] = (uint32_t)a.dp[pe] + (uint32_t)a.dq[qe];
                    coff[e] = bil ? (uint32_t)a.cp[pe] + (uint32_t)a.cq[qe] : 0u;
                }
                d_run = d_run && doff[e] == doff[0] + (uint32_t)e;
                c_run = c_run && coff[e] == coff[0] + (uint32_t)e;
                if(++q == a.Q)
                {
                    q = 0;
                    p++;
                }
            }
            if(bil)
            {
                if(c_run)
                    __builtin_memcpy(&c, (const E*)a.C + coff[0], sizeof(c));
                else
                {
#pragma unroll
                    for(int e = 0; e < V; e++)
                        c.v[e] = ((const E*)a.C)[coff[e]];
                }
            }
            const O* src = (const O*)a.ws + (size_t)z0 * total + (idx - over);
            Vec      s   = {};
            auto     add = [&](const Vec& x) {
#pragma unroll
                for(int e = 0; e < V; e++)
                    s.v[e] = Fin::add(s.v[e], x.v[e]);
            };
            auto take = [&](auto width, int z) {
                constexpr int W = decltype(width)::value;
                Vec           x[W];
#pragma unroll
                for(int u = 0; u < W; u++)
                    __builtin_memcpy(&x[u], src + (size_t)(z + u) * total, sizeof(Vec));
                if(z == 0)
                    s = x[0];
                else
                    add(x[0]);
#pragma unroll
                for(int u = 1; u < W; u++)
                    add(x[u]);
            };
            int z = 0;
            for(; z + DEPTH <= n; z += DEPTH)
                take(std::integral_constant<int, DEPTH>{}, z);
            if(DEPTH > 4 && z + 4 <= n) // (fewer than DEPTH are left)
            {
                take(std::integral_constant<int, 4>{}, z);
                z += 4;
            }
            if(z + 2 <= n)
            {
                take(std::integral_constant<int, 2>{}, z);
                z += 2;
            }
            if(z < n)
                take(std::integral_constant<int, 1>{}, z);
            if constexpr(DEALT)
            {
                __shared__ Vec part[256];
                part[threadIdx.x] = s;
                __syncthreads();
                if(g != 0 || !in)
                    return;
                for(int h = 1; h < 256 >> lane_bits && h * per < a.split_k; h++)
                    add(part[(h << lane_bits) + lane]);
            }
            // the last vector's outputs back to the front
#pragma unroll
            for(int h = 1; h < V; h++)
                if(over >= h)
                {
#pragma unroll
                    for(int e = 0; e + 1 < V; e++)
                        s.v[e] = s.v[e + 1];
                }
            Elems d;
#pragma unroll
            for(int e = 0; e < V; e++)
                d.v[e] = Fin::finish(s.v[e], a.alpha, a.beta, bil, &c.v[e]);
            if(d_run)
                __builtin_memcpy((E*)a.D + doff[0], &d, sizeof(d));
            else
            {
#pragma unroll
                for(int e = 0; e < V; e++)
                    if(idx + e < total)
                        ((E*)a.D)[doff[e]] = d.v[e];
            }
        }

        template <typename Fin>
        int launch_reduce(const KArgs& a, hipStream_t stream)
        {
            constexpr int V     = sizeof(typename Fin::O) >= 16 ? 1 : 16 / (int)sizeof(typename Fin::O);
            const size_t  total = (size_t)a.P * (size_t)a.Q;
            // 16 bytes a thread once that still puts eight wavefronts on every compute unit, if the outputs are one run of
            // D after another (f32 1450 x 1450 in 4 slices 7.3 us, one output a thread 8.4; with offsets from tables, of
            // which a thread then has V to wait for, 2048 x 2048 in 2 17.4 and 14.2)
            if(V > 1 && total >= (size_t)V * 131072 && a.cd_affine && a.dq_stride == 1)
            {
                const size_t blocks = (total + 256 * V - 1) / (256 * V);
                hipLaunchKernelGGL((splitk_reduce_kernel<Fin, V, false, 4>), dim3((unsigned)blocks), dim3(256), 0, stream, a, 8, a.split_k);
                return (int)hipGetLastError();
            }
            // four 16-byte loads or eight smaller ones in flight: more from slices that lie a power of two apart meet in the
            // same channels (f32 1024 x 1024 in 16 slices 12.3 us against 13.6 with eight of 16 bytes, c64 512 x 512 in 16
            // 11.9 and 13.4), fewer wait (f32 700 x 750 in 16, four of 4 bytes 8.0, eight 6.8)
            constexpr int DEPTH = sizeof(typename Fin::O) >= 16 ? 4 : 8;
            // threads enough for eight wavefronts a compute unit, at least four slices each
            int lane_bits = 8;
            while(lane_bits > 3 && (total << (8 - lane_bits)) < 131072 && (a.split_k >> (9 - lane_bits)) >= 4)
                lane_bits--;
            const int    groups = 256 >> lane_bits, per = (a.split_k + groups - 1) / groups;
            const size_t blocks = (total + ((size_t)1 << lane_bits) - 1) >> lane_bits;
            if(groups > 1)
                hipLaunchKernelGGL((splitk_reduce_kernel<Fin, 1, true, DEPTH>), dim3((unsigned)blocks), dim3(256), 0, stream, a, lane_bits, per);
            else
                hipLaunchKernelGGL((splitk_reduce_kernel<Fin, 1, false, DEPTH>), dim3((unsigned)blocks), dim3(256), 0, stream, a, lane_bits, per);
            return (int)hipGetLastError();
        }

        int reduce_dispatch(int cls, const KArgs& a, hipStream_t stream)
        {
            switch(cls)
            {
            case HIPTK_F16: return launch_reduce<FinF16>(a, stream);
            case HIPTK_BF16: return launch_reduce<FinBF16>(a, stream);
            case HIPTK_F32:
            case HIPTK_F32_AS_F16:
            case HIPTK_F32_AS_BF16: return launch_reduce<FinWide<WTraitsF32>>(a, stream);
            case HIPTK_F64: return launch_reduce<FinWide<WTraitsF64>>(a, stream);
            case HIPTK_C32: return launch_reduce<FinWide<WTraitsC32>>(a, stream);
            case HIPTK_C64: return launch_reduce<FinWide<WTraitsC64>>(a, stream);
            case HIPTK_F64_AS_F32: return launch_reduce<FinWide<WTraitsF64AsF32>>(a, stream);
            default: return (int)hipErrorInvalidValue;
            }
        }

        // What the 16-byte vectors of a direct-load kernel must start at multiples of, bytes
        int vec_align(const KernelEntry& e)
        {
            return e.vec_align ? e.vec_align : 16;
        }
        // ... and what a problem's do (1, as a flag: 16)
        int xy_aligned(const hiptk_problem_t* p)
        {
            return p->xy_aligned == 1 ? 16 : p->xy_aligned;
        }

        // The affine-K variant is preferred when the problem allows it; the table variant
        // serves every problem.
        const KernelEntry* find_entry(const hiptk_problem_t* p)
        {
            const KernelEntry* table = nullptr;
            for(const KernelEntry& e : registry().all)
            {
                if(e.cls == p->cls && e.tile_id == p->tile_id && e.x_kfast == (p->x_kfast != 0)
                   && e.y_kfast == (p->y_kfast != 0) && e.x_vec == p->x_vec && e.y_vec == p->y_vec)
                {
                    // a tile can only be moved back to end at P / Q if it fits into P / Q
                    if((p->shift_p && p->P < e.bp) || (p->shift_q && p->Q < e.bq))
                        continue;
                    // the direct-load kernels: a restricted K tail, vectors on multiples of 16 (or 4) bytes
                    if(e.k_multiple > 0 && (p->K % e.k_multiple != 0 || p->K < e.bk || xy_aligned(p) < vec_align(e)))
                        continue;
                    // ... and they address an operand with 32-bit byte offsets
                    if(e.k_multiple > 0)
                    {
                        const uint64_t eb   = (uint64_t)operand_bytes(p->cls);
                        const int32_t  most = p->x_max_off > p->y_max_off ? p->x_max_off : p->y_max_off;
                        // (less the bias some of them keep in a lane's offset so that loads can share a write of M0)
                        if(most < 0 || ((uint64_t)most + 16 / eb) * eb > 0xFFFFFFFFull - (uint64_t)DMA_BIAS)
                            continue;
                    }
                    if(e.k_affine && p->k_affine)
                        return &e;
                    if(!e.k_affine && !table)
                        table = &e;
                }
            }
            return table;
        }

        // What runs in place of a direct-load kernel when an operand's base address is not aligned for it: the
        // register-staged tile the problem names, else the largest one of its class and layout.
        const KernelEntry* staged_entry(const hiptk_problem_t* p)
        {
            const KernelEntry* best = nullptr;
            hiptk_problem_t    q    = *p;
            if(p->unaligned_split > 0)
            {
                q.tile_id            = p->unaligned_tile;
                const KernelEntry* e = find_entry(&q);
                if(e && e->k_multiple == 0)
                    return e;
            }
            for(const KernelEntry& t : registry().all)
            {
                if(t.cls != p->cls || t.k_multiple > 0)
                    continue;
                q.tile_id            = t.tile_id;
                const KernelEntry* e = find_entry(&q);
                if(e && e->k_multiple == 0
                   && (!best || e->bp * e->bq > best->bp * best->bq
                       || (e->bp * e->bq == best->bp * best->bq && e->threads > best->threads)))
                    best = e;
            }
            return best;
        }

        // The entry a launch with these operand addresses runs: the resolved one where the plan
        // resolved it (and the problem still is the one it was resolved for), else a search.  stands_in: it is
        // not the plan's tile, but what runs for operands that are not aligned for that.
        const KernelEntry* entry_for(const hiptk_problem_t* p, const void* X, const void* Y, bool& stands_in)
        {
            const KernelEntry* e = (const KernelEntry*)p->kernel;
            const bool         resolved = e && e->cls == p->cls && e->tile_id == p->tile_id && e->x_kfast == (p->x_kfast != 0)
                                  && e->y_kfast == (p->y_kfast != 0) && e->x_vec == p->x_vec && e->y_vec == p->y_vec;
            if(!resolved)
                e = find_entry(p);
            stands_in = e && e->k_multiple > 0 && ((((uintptr_t)X) | ((uintptr_t)Y)) & (uintptr_t)(vec_align(*e) - 1)) != 0;
            if(stands_in)
                e = resolved ? (const KernelEntry*)p->kernel_unaligned : staged_entry(p);
            return e;
        }
    }
}

extern "C" int hiptk_resolve(hiptk_problem_t* prob)
{
    if(!prob)
        return HIPTK_ERR_ARG;
    const hiptk::KernelEntry* e = hiptk::find_entry(prob);
    prob->kernel                = e;
    prob->kernel_unaligned      = (e && e->k_multiple > 0) ? hiptk::staged_entry(prob) : e;
    return e ? HIPTK_OK : HIPTK_ERR_NO_KERNEL;
}

extern "C" const char* hiptk_kernel_name_at(const hiptk_problem_t* prob, const void* X, const void* Y)
{
    bool                      stands_in;
    const hiptk::KernelEntry* e = prob ? hiptk::entry_for(prob, X, Y, stands_in) : nullptr;
    return e ? e->name : "";
}

extern "C" int hiptk_tile_count(int cls)
{
    int n = 0;
    for(const hiptk::KernelEntry& e : hiptk::registry().all)
        if(e.cls == cls && e.tile_id + 1 > n)
            n = e.tile_id + 1;
    return n;
}

extern "C" int hiptk_tile_info(int cls, int tile_id, hiptk_tile_info_t* out)
{
    if(!out)
        return HIPTK_ERR_ARG;
    for(const hiptk::KernelEntry& e : hiptk::registry().all)
    {
        if(e.cls == cls && e.tile_id == tile_id)
        {
            out->tile_id   = tile_id;
            out->bp        = e.bp;
            out->bq        = e.bq;
            out->bk        = e.bk;
            out->threads   = e.threads;
            out->lds_bytes = e.lds_bytes;
            out->k_multiple = e.k_multiple;
            out->mfma_k     = e.mfma_k;
            out->vec_align  = e.k_multiple > 0 ? hiptk::vec_align(e) : 0;
            std::snprintf(out->name, sizeof(out->name), "cls%d_%dx%dx%d", cls, e.bp, e.bq, e.bk);
            return HIPTK_OK;
        }
    }
    return HIPTK_ERR_NO_KERNEL;
}

extern "C" int hiptk_kernel_available(const hiptk_problem_t* prob)
{
    return (prob && hiptk::find_entry(prob)) ? 1 : 0;
}

extern "C" const char* hiptk_kernel_name(const hiptk_problem_t* prob)
{
    const hiptk::KernelEntry* e = prob ? hiptk::find_entry(prob) : nullptr;
    return e ? e->name : "";
}

extern "C" uint64_t hiptk_workspace_bytes(const hiptk_problem_t* prob)
{
    if(!prob || prob->split_k <= 1)
        return 0;
    return (uint64_t)prob->split_k * (uint64_t)prob->P * (uint64_t)prob->Q
           * (uint64_t)hiptk::acc_bytes(prob->cls);
}

// Many long slices: an XCD takes whole slices, whose tiles read the same panels, instead of a band of every
// slice's tiles, where each panel went to all eight L2s (bf16 324 x 207 x 52974 in 32 slices 40.8 -> 23.4 us, f64
// 116 x 144 x 54844 in 16 87.0 -> 66.8, f32 256 x 256 x 65536 in 32 76.5 -> 71.8).  Few or short slices start on
// cold panels all at once, and the tiles of one wait on the same lines: 1.00-1.11 of the time (c32 320 x 768 x 128
// in 4 11.2 -> 12.4, bf16 1024 x 224 x 800 in 8 18.7 -> 19.4).
extern "C" int hiptk_slices_by_die(int64_t ktiles, int64_t split)
{
    if(ktiles < 1 || split < 1)
        return 0;
    const int64_t per    = (ktiles + split - 1) / split;
    const int64_t slices = (ktiles + per - 1) / per;
    return slices >= 8 && slices * per >= 160;
}

extern "C" int hiptk_contract(const hiptk_problem_t* prob,
                              const void*            alpha,
                              const void*            beta,
                              const void*            X,
                              const void*            Y,
                              const void*            C,
                              void*                  D,
                              void*                  workspace,
                              uint64_t               workspace_bytes,
                              void*                  stream,
                              int*                   hip_error)
{
    using namespace hiptk;
    if(hip_error)
        *hip_error = 0;
    if(!prob || !alpha || !X || !Y || !D)
        return HIPTK_ERR_ARG;
    if(prob->P <= 0 || prob->Q <= 0 || prob->K <= 0 || prob->P > 0x7FFFFF00ll || prob->Q > 0x7FFFFF00ll
       || prob->K > 0x7FFFFF00ll || prob->split_k < 1)
        return HIPTK_ERR_ARG;
    if(!prob->xp || !prob->xk || !prob->yq || !prob->yk || !prob->dp || !prob->dq)
        return HIPTK_ERR_ARG;
    const bool bil = prob->op == HIPTK_OP_BILINEAR;
    if(bil && (!C || !beta || !prob->cp || !prob->cq))
        return HIPTK_ERR_ARG;
    bool               stands_in = false;
    const KernelEntry* e         = entry_for(prob, X, Y, stands_in);
    if(!e)
        return HIPTK_ERR_NO_KERNEL;

    KArgs a;
    std::memset(&a, 0, sizeof(a));
    a.X  = X;
    a.Y  = Y;
    a.C  = C;
    a.D  = D;
    a.ws = workspace;
    a.xp = prob->xp;
    a.xk = prob->xk;
    a.yq = prob->yq;
    a.yk = prob->yk;
    a.cp = prob->cp;
    a.cq = prob->cq;
    a.dp = prob->dp;
    a.dq = prob->dq;
    a.P  = (int32_t)prob->P;
    a.Q  = (int32_t)prob->Q;
    a.K  = (int32_t)prob->K;
    a.bilinear  = bil ? 1 : 0;
    a.cd_affine = prob->cd_affine;
    a.dp_stride = prob->dp_stride;
    a.dq_stride = prob->dq_stride;
    a.cp_stride = prob->cp_stride;
    a.cq_stride = prob->cq_stride;
    a.xp_stride = prob->cd_affine ? prob->xp_stride : 0;
    a.yq_stride = prob->cd_affine ? prob->yq_stride : 0;
    a.xk_stride = prob->xk_stride;
    a.yk_stride = prob->yk_stride;
    a.cd_vec    = prob->cd_vec;
    a.shift_p   = prob->shift_p ? 1 : 0;
    a.shift_q   = prob->shift_q ? 1 : 0;
    {
        // byte offset of the last 16-byte vector of X / Y (the class's own element size)
        const int32_t eb = operand_bytes(prob->cls), back = 16 / eb - 1;
        a.x_last_vec     = prob->x_max_off >= back ? (uint32_t)eb * (uint32_t)(prob->x_max_off - back) : 0u;
        a.y_last_vec     = prob->y_max_off >= back ? (uint32_t)eb * (uint32_t)(prob->y_max_off - back) : 0u;
    }
    a.x_chunked = (prob->x_kfast && prob->x_rows_adjacent) ? 1 : 0;
    a.y_chunked = (prob->y_kfast && prob->y_rows_adjacent) ? 1 : 0;
    // A moved-back tile stores whole 8-element vectors of D that reach into its neighbour's
    // columns (same values).  When D is updated in place (C == D) the neighbour's elements must
    // not be read and written twice, so that case stores element by element.
    if(a.shift_q && bil && C == D && prob->Q % 8 != 0)
        a.cd_vec = 1;
    a.tiles_p  = (int32_t)((prob->P + e->bp - 1) / e->bp);
    a.tiles_q  = (int32_t)((prob->Q + e->bq - 1) / e->bq);
    const int ktiles = (int)((prob->K + e->bk - 1) / e->bk);
    int       split  = prob->split_k;
    if(stands_in && prob->unaligned_split > 0)
    {
        // (its slices may want more workspace than the plan asked for)
        const uint64_t slice = (uint64_t)prob->P * (uint64_t)prob->Q * (uint64_t)acc_bytes(prob->cls);
        const uint64_t held  = workspace ? workspace_bytes / slice : 0;
        split                = held < (uint64_t)prob->unaligned_split ? std::max(1, (int)held) : prob->unaligned_split;
    }
    if(split > ktiles)
        split = ktiles;
    a.ktiles_per_split = (ktiles + split - 1) / split;
    split              = (ktiles + a.ktiles_per_split - 1) / a.ktiles_per_split; // no empty slice
    a.split_k          = split;
    a.slice_bands = hiptk_slices_by_die(ktiles, split) && (uint64_t)a.tiles_p * (uint64_t)a.tiles_q * (uint64_t)split <= 0x7FFFFFFFull
                        ? 1
                        : 0;
    if((uint64_t)a.tiles_p * (uint64_t)a.tiles_q > 0x7FFFFFFFull || split > 65535)
        return HIPTK_ERR_ARG;

    switch(prob->cls)
    {
    case HIPTK_C32:
        a.alpha[0] = ((const float*)alpha)[0];
        a.alpha[1] = ((const float*)alpha)[1];
        if(beta)
        {
            a.beta[0] = ((const float*)beta)[0];
            a.beta[1] = ((const float*)beta)[1];
        }
        break;
    case HIPTK_C64:
        a.alpha[0] = ((const double*)alpha)[0];
        a.alpha[1] = ((const double*)alpha)[1];
        if(beta)
        {
            a.beta[0] = ((const double*)beta)[0];
            a.beta[1] = ((const double*)beta)[1];
        }
        break;
    case HIPTK_F64:
    case HIPTK_F64_AS_F32:
        a.alpha[0] = *(const double*)alpha;
        if(beta)
            a.beta[0] = *(const double*)beta;
        break;
    default:
        a.alpha[0] = *(const float*)alpha;
        if(beta)
            a.beta[0] = *(const float*)beta;
        break;
    }

    if(split > 1)
    {
        const uint64_t need
            = (uint64_t)split * (uint64_t)prob->P * (uint64_t)prob->Q * (uint64_t)acc_bytes(prob->cls);
        if(!workspace || workspace_bytes < need)
            return HIPTK_ERR_WORKSPACE;
    }

    hipStream_t s  = (hipStream_t)stream;
    int         rc = e->launch(a, s);
    if(rc == 0 && split > 1)
        rc = reduce_dispatch(prob->cls, a, s);
    if(rc != 0)
    {
        if(hip_error)
            *hip_error = rc;
        return HIPTK_ERR_LAUNCH;
    }
    return HIPTK_OK;
}

// ---- a workspace that lives in the library, for callers that cannot allocate ----
//
// Device memory of a fixed, modest size that every device the library runs on holds until the
// process ends.  In host code the array's name is only a stand-in (passing it to a kernel would
// hand the kernel a host-side address); its device address is looked up once per device with
// hipGetSymbolAddress, with that device current, and from then on only that address is used.
static __device__ __align__(256) unsigned char scratch[HIPTK_STATIC_WORKSPACE_BYTES];

namespace
{
    constexpr int MAX_DEVICES = 64;
    std::mutex    g_scratch_lock;
    void*         g_scratch_ptr[MAX_DEVICES] = {};
}

extern "C" int hiptk_static_workspace(void** ptr, uint64_t* bytes, int* hip_error)
{
    if(hip_error)
        *hip_error = 0;
    if(!ptr || !bytes)
        return HIPTK_ERR_ARG;
    *ptr   = nullptr;
    *bytes = 0;
    int        dev = -1;
    hipError_t e   = hipGetDevice(&dev);
    if(e != hipSuccess || dev < 0 || dev >= MAX_DEVICES)
    {
        if(hip_error)
            *hip_error = (int)e;
        return HIPTK_ERR_LAUNCH;
    }
    std::lock_guard<std::mutex> guard(g_scratch_lock);
    if(!g_scratch_ptr[dev])
    {
        void* p = nullptr;
        e       = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        if(e != hipSuccess || !p)
        {
            if(hip_error)
                *hip_error = (int)e;
            return HIPTK_ERR_LAUNCH;
        }
        g_scratch_ptr[dev] = p;
    }
    *ptr   = g_scratch_ptr[dev];
    *bytes = HIPTK_STATIC_WORKSPACE_BYTES;
    return HIPTK_OK;
}
