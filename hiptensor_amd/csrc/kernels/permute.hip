// Tensor permutation kernels, B[perm(index)] = opB(alpha * opA(A[index])), and their launcher.
//
// The work is a stream of bytes through HBM, so the kernels are built around memory
// coalescing, not arithmetic:
//   * COPY    one fused mode left: a scaled vector copy.
//   * TILED   A's fastest mode i and B's fastest mode j differ.  A workgroup moves a
//             two-dimensional tile of those two modes: it reads rows along i (contiguous in A),
//             applies the element operation, parks the tile in LDS, and writes it out along j
//             (contiguous in B).  The other modes only choose the tile's base offsets, once per
//             workgroup on the scalar unit.
//   * ROWS    A and B share the fastest mode: runs of it are contiguous on both sides and go
//             from registers straight back to memory, no LDS.
//   * STRIP   like TILED, for a tile mode too short to give long runs (the 3 of an RGB image,
//             say) when the other tile mode follows it directly in memory on that side: a
//             workgroup takes a strip of the long mode times the whole short mode, which is one
//             contiguous run on the short mode's side, and moves it linearly there.
//   * GROUPED TILED for tensors of many short modes: a tile row spans A's two fastest modes, a
//             tile column B's two fastest modes, so that runs stay long when no single mode is.
//   * SHARED  ROWS for a short shared fastest mode (interleaved channels): tiles of that mode
//             times a chunk of A's next mode times a chunk of B's next mode, through LDS.
//   * RUNS    ROWS without tiles: B is written front to back in 16-byte vectors, each thread finding
//             where its vector's run lies in A; for runs that no tile covers well or whose odd
//             length leaves ROWS only narrow vectors.
//   * GATHER  one thread per element of B; covers tiny tensors and awkward extents.
// Element operation per Composable Kernel's UnaryCombinedOp<Aop, Scale, Bop>
// (ck/tensor_operation/gpu/element/combined_element_wise_operation.hpp:14-32): every step is
// rounded to the element type; for f16 alpha is rounded to half first
// (unary_element_wise_operation.hpp:647-651).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <type_traits>

#include "hiptk_kernels.h"
#include "perm_addr.hpp"

namespace hiptk
{
    namespace
    {

        struct PArgs
        {
            const void* A;
            void*       B;
            uint32_t    e_i, e_j; // extents of the two tile modes
            uint32_t    a_j; // A stride of mode j (mode i has stride 1 in A)
            uint32_t    b_i, b_j; // B strides (TILED: b_j == 1, ROWS: b_i == 1)
            uint32_t    nt_i, nt_j; // tiles along i and j
            uint32_t    group; // tile order: bands of `group` tiles along j, walked j-first
            int32_t     bands; // 1: each die takes neighbouring tiles (tile_work)
            int32_t     keep; // 1: ordinary stores, so that the caches put lines of two tiles together
            int32_t     nb; // modes that only pick the tile's base
            uint32_t    bext[PERM_BATCH], ba[PERM_BATCH], bb[PERM_BATCH];
            float       alpha;
            int32_t     op_a, op_b;
        };

        struct GArgs
        {
            const void* A;
            void*       B;
            uint32_t    n;
            int32_t     rank;
            uint32_t    ext[HIPTK_PERM_MAX_RANK]; // in B's order, fastest first; extents of 1 left out
            uint32_t    astr[HIPTK_PERM_MAX_RANK];
            uint32_t    magic[HIPTK_PERM_MAX_RANK]; // floor(2^32 / ext) + 1
            float       alpha;
            int32_t     op_a, op_b;
        };

        template <typename T, int V>
        struct alignas(sizeof(T) * V) Vec
        {
            T v[V];
        };

        // Every element is read once and written once: loads and stores are marked non-temporal so
        // that the stream does not displace itself in the caches (measured: a plain 1 GiB copy
        // 5.8 TB/s, with non-temporal loads and stores 6.2 TB/s).
        template <int BYTES>
        struct RawBits;
        template <>
        struct RawBits<2>
        {
            using type = uint16_t;
        };
        template <>
        struct RawBits<4>
        {
            using type = uint32_t;
        };
        template <>
        struct RawBits<8>
        {
            using type = uint32_t __attribute__((ext_vector_type(2)));
        };
        template <>
        struct RawBits<16>
        {
            using type = uint32_t __attribute__((ext_vector_type(4)));
        };

        template <typename T, int V>
        __device__ inline Vec<T, V> load_stream(const T* p)
        {
            using R = typename RawBits<sizeof(T) * V>::type;
            const R r = __builtin_nontemporal_load(reinterpret_cast<const R*>(p));
            return __builtin_bit_cast(Vec<T, V>, r);
        }

        template <typename T, int V>
        __device__ inline void store_stream(T* p, const Vec<T, V>& v)
        {
            using R = typename RawBits<sizeof(T) * V>::type;
            __builtin_nontemporal_store(__builtin_bit_cast(R, v), reinterpret_cast<R*>(p));
        }

        // 16 bytes at any multiple of the element
        template <int ALIGN>
        struct LooseBits;
        template <>
        struct LooseBits<2>
        {
            typedef uint32_t type __attribute__((ext_vector_type(4), aligned(2)));
        };
        template <>
        struct LooseBits<4>
        {
            typedef uint32_t type __attribute__((ext_vector_type(4), aligned(4)));
        };

        template <typename T>
        __device__ inline Vec<T, 16 / (int)sizeof(T)> load_loose(const T* p)
        {
            using R = typename LooseBits<sizeof(T)>::type;
            return __builtin_bit_cast(Vec<T, 16 / (int)sizeof(T)>, __builtin_nontemporal_load(reinterpret_cast<const R*>(p)));
        }

        template <typename T>
        __device__ inline void store_loose(T* p, const Vec<T, 16 / (int)sizeof(T)>& v)
        {
            using R = typename LooseBits<sizeof(T)>::type;
            __builtin_nontemporal_store(__builtin_bit_cast(R, v), reinterpret_cast<R*>(p));
        }

        template <typename T>
        __device__ inline T element_op(T x, T alpha, int op_a, int op_b)
        {
            if(op_a == HIPTK_PERM_OP_RAW)
                return x; // a plain move: every bit pattern, NaN payloads included, arrives unchanged
            T y = x;
            if(op_a)
                y = y * y;
            y = alpha * y;
            if(op_b)
                y = y * y;
            return y;
        }

        // Bound by HBM where runs are whole lines, and by the number of accesses and by lines written in two parts where they
        // are not.  LOOSE: 16-byte vectors at any element on both sides.  `bands` and `keep` (set by the planner, with the
        // reasons): tiles that share lines meet in one cache, which puts the lines together.  The three together, f16
        // 1943.205.637 -> (2,1,0) 510 -> 262 us, 505.606.133 -> (2,0,1) 104 -> 39, f32 946.579.437 -> (2,1,0) 762 -> 483; bands
        // alone, f32 1 GiB in whole lines 376 -> 367.5 (5.84 TB/s).
        // The tile in LDS is [TJ][TI].  Column reads must spread over the 64 banks: the small
        // tiles pad each row by one element; the 64 KiB tiles have no room for padding and XOR
        // the column index with the row number instead (in units of one 32-bit word).
        template <typename T, int TI, int TJ, int VR, int VW, bool TRANSPOSE, bool LOOSE = false, int NT = PERM_THREADS, bool SWZ = false>
        __global__ __launch_bounds__(NT) void permute_tile_kernel(PArgs a)
        {
            constexpr int PITCH = SWZ ? TI : TI + 4 / (int)sizeof(T); // an odd number of 32-bit words
            constexpr int VPR   = TI / VR; // vectors per tile row
            constexpr int NRV   = VPR * TJ / NT; // vectors per thread, read side
            static_assert(TI % VR == 0 && (VPR * TJ) % NT == 0 && NRV >= 1, "read shape");
            static_assert(!SWZ || TI * sizeof(T) >= 256, "a swizzled row spans all 64 banks");
            static_assert(!LOOSE || TRANSPOSE, "rows have the linear kernel for that");
            __shared__ T tile[TRANSPOSE ? TJ * PITCH : 1];
            auto         at = [](uint32_t j, uint32_t i) -> uint32_t {
                return SWZ ? j * TI + (i ^ ((j & 63u) * (4u / sizeof(T)))) : j * PITCH + i;
            };

            const T* __restrict__ A = static_cast<const T*>(a.A);
            T* __restrict__ B       = static_cast<T*>(a.B);
            const int tid           = threadIdx.x;

            uint32_t i0, j0, aoff, boff;
            tile_origin(a, tile_work(blockIdx.x, gridDim.x, a.bands != 0), TI, TJ, i0, j0, aoff, boff);
            // the part of the tile inside the extents
            const uint32_t nx = a.e_i - i0 < TI ? a.e_i - i0 : TI, ny = a.e_j - j0 < TJ ? a.e_j - j0 : TJ;

            const T alpha = static_cast<T>(a.alpha);

            if(!LOOSE || nx >= VR)
            {
                Vec<T, VR> r[NRV];
#pragma unroll
                for(int k = 0; k < NRV; ++k)
                {
                    // Lanes outside the extents load the tile's first element instead of branching
                    // around the load: a branch per load would make the compiler wait for each load
                    // before issuing the next, and the loads must all be in flight together.
                    const TileVector v    = tile_vector<VR, LOOSE>(tid + k * NT, VPR, nx, ny);
                    const T*         from = A + aoff + (v.ok ? v.at + v.line * a.a_j : 0u);
                    if constexpr(LOOSE)
                        r[k] = load_loose(from);
                    else
                        r[k] = load_stream<T, VR>(from);
                }
#pragma unroll
                for(int k = 0; k < NRV; ++k)
                {
                    const TileVector v = tile_vector<VR, LOOSE>(tid + k * NT, VPR, nx, ny);
#pragma unroll
                    for(int e = 0; e < VR; ++e)
                        r[k].v[e] = element_op(r[k].v[e], alpha, a.op_a, a.op_b);
                    if constexpr(TRANSPOSE)
                    {
                        if(!LOOSE || v.ok)
#pragma unroll
                            for(int e = 0; e < VR; ++e)
                                tile[at(v.line, v.at + e)] = r[k].v[e];
                    }
                    else
                    {
                        if(v.ok)
                            store_stream<T, VR>(B + boff + v.at + v.line * a.b_j, r[k]);
                    }
                }
            }
            else
            {
                // (the last tile of an extent that leaves it less than a vector)
                for(uint32_t u = tid; u < nx * ny; u += NT)
                    tile[at(u / nx, u % nx)] = element_op(A[aoff + u % nx + u / nx * a.a_j], alpha, a.op_a, a.op_b);
            }
            if constexpr(TRANSPOSE)
            {
                constexpr int VPC = TJ / VW; // vectors per tile column
                constexpr int NWV = VPC * TI / NT;
                static_assert(TJ % VW == 0 && (VPC * TI) % NT == 0 && NWV >= 1, "write shape");
                __syncthreads();
                auto write = [&](auto keep_c) {
#pragma unroll
                    for(int k = 0; k < NWV; ++k)
                    {
                        const TileVector v = tile_vector<VW, LOOSE>(tid + k * NT, VPC, ny, nx);
                        Vec<T, VW>       o;
#pragma unroll
                        for(int e = 0; e < VW; ++e)
                            o.v[e] = tile[at(v.at + e, v.line)];
                        T* to = B + boff + v.at + v.line * a.b_i;
                        if(v.ok)
                        {
                            if constexpr(decltype(keep_c)::value)
                                __builtin_memcpy(to, &o, sizeof(o));
                            else if constexpr(LOOSE)
                                store_loose(to, o);
                            else
                                store_stream<T, VW>(to, o);
                        }
                    }
                };
                if(LOOSE && ny < VW)
                {
                    for(uint32_t u = tid; u < nx * ny; u += NT)
                        B[boff + u % ny + u / ny * a.b_i] = tile[at(u % ny, u / ny)];
                }
                else if(a.keep)
                    write(std::integral_constant<bool, true>{});
                else
                    write(std::integral_constant<bool, false>{});
            }
        }

        struct SArgs
        {
            const void* A;
            void*       B;
            uint32_t    e_s, e_l; // extents of the short and of the long tile mode
            uint32_t    row_stride; // stride of the short mode on the side that is walked in rows
            uint32_t    magic; // floor(2^32 / e_s) + 1: v / e_s == umulhi(v, magic) for v < 2^28
            uint32_t    nt; // strips along the long mode
            int32_t     nb;
            uint32_t    bext[PERM_BATCH], ba[PERM_BATCH], bb[PERM_BATCH];
            float       alpha;
            int32_t     op_a, op_b;
        };

        // LINEAR_WRITE: the long mode is A's fastest, the short one B's fastest, and B holds the
        // long mode right after the short one, so a strip is one run of cnt * e_s elements of B.
        // It is read in e_s rows of A and written linearly.  !LINEAR_WRITE is the mirror image:
        // the short mode is A's fastest with the long one right after it; the strip is read
        // linearly from A and written in e_s rows of B.
        // Position of a linear index v of a strip: v = x * e_s + s.  One division per thread finds
        // the first position; afterwards the walk only adds (32-bit integer multiplies and
        // divides run at a quarter of the add rate, and this kernel has one per element to spare).
        struct StripPos
        {
            uint32_t s, x;
            __device__ void advance(uint32_t ds, uint32_t dx, uint32_t e_s)
            {
                s += ds;
                x += dx;
                if(s >= e_s)
                {
                    s -= e_s;
                    ++x;
                }
            }
        };

        template <typename T, int TL, int VL, int VS, bool LINEAR_WRITE>
        __global__ __launch_bounds__(PERM_THREADS) void permute_strip_kernel(SArgs a)
        {
            constexpr int NT    = PERM_THREADS;
            constexpr int U     = 8; // loads in flight per thread: a whole 32 KiB strip of full vectors
            constexpr int PITCH = TL + 4 / (int)sizeof(T); // an odd number of 32-bit words: rows start in different banks
            constexpr int VPR   = TL / VS; // row vectors per strip row
            static_assert(TL % VS == 0 && TL % VL == 0, "strip shape");
            extern __shared__ unsigned char strip_smem[];
            T* tile = reinterpret_cast<T*>(strip_smem); // [e_s][PITCH]

            const T* __restrict__ A = static_cast<const T*>(a.A);
            T* __restrict__ B       = static_cast<T*>(a.B);
            const uint32_t tid      = threadIdx.x;

            uint32_t       blk = blockIdx.x;
            const uint32_t t   = blk % a.nt;
            blk /= a.nt;
            uint32_t aoff = 0, boff = 0;
            for(int d = 0; d < a.nb; ++d)
            {
                const uint32_t c = blk % a.bext[d];
                blk /= a.bext[d];
                aoff += c * a.ba[d];
                boff += c * a.bb[d];
            }
            const uint32_t l0  = t * TL;
            const uint32_t cnt = (a.e_l - l0) < (uint32_t)TL ? (a.e_l - l0) : (uint32_t)TL;
            const T        alpha = static_cast<T>(a.alpha);
            const uint32_t nrv   = a.e_s * VPR; // row vectors of the strip (tail rows included)
            const uint32_t nlv   = cnt * a.e_s / VL; // linear vectors of the strip

            // the walk over linear vectors u = tid, tid + NT, ...: first element v = u * VL
            StripPos pos;
            pos.x = __umulhi(tid * VL, a.magic);
            pos.s = tid * VL - pos.x * a.e_s;
            const uint32_t step_x = __umulhi((uint32_t)(NT * VL), a.magic); // scalar
            const uint32_t step_s = NT * VL - step_x * a.e_s;

            if constexpr(LINEAR_WRITE)
            {
                aoff += l0;
                boff += l0 * a.e_s;
                for(uint32_t u0 = 0; u0 < nrv; u0 += NT * U)
                {
                    Vec<T, VS> r[U];
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        // out-of-range lanes load the strip's first element (no branch: see the tile kernel)
                        const uint32_t u = u0 + tid + k * NT, s = u / VPR, xv = u % VPR;
                        const bool     ok = u < nrv && xv * VS < cnt;
                        r[k] = load_stream<T, VS>(A + aoff + (ok ? xv * VS + s * a.row_stride : 0u));
                    }
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        const uint32_t u = u0 + tid + k * NT, s = u / VPR, xv = u % VPR;
                        if(u < nrv)
                        {
#pragma unroll
                            for(int e = 0; e < VS; ++e)
                                tile[s * PITCH + xv * VS + e] = element_op(r[k].v[e], alpha, a.op_a, a.op_b);
                        }
                    }
                }
                __syncthreads();
                for(uint32_t u = tid; u < nlv; u += NT)
                {
                    Vec<T, VL> o;
                    StripPos   q = pos;
#pragma unroll
                    for(int e = 0; e < VL; ++e)
                    {
                        o.v[e] = tile[q.s * PITCH + q.x];
                        q.advance(1, 0, a.e_s);
                    }
                    store_stream<T, VL>(B + boff + u * VL, o);
                    pos.advance(step_s, step_x, a.e_s);
                }
            }
            else
            {
                aoff += l0 * a.e_s;
                boff += l0;
                for(uint32_t u0 = 0; u0 < nlv; u0 += NT * U)
                {
                    Vec<T, VL> r[U];
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        const uint32_t u = u0 + tid + k * NT;
                        r[k] = load_stream<T, VL>(A + aoff + (u < nlv ? u * VL : 0u));
                    }
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        const uint32_t u = u0 + tid + k * NT;
                        if(u < nlv)
                        {
                            StripPos q = pos;
#pragma unroll
                            for(int e = 0; e < VL; ++e)
                            {
                                tile[q.s * PITCH + q.x] = element_op(r[k].v[e], alpha, a.op_a, a.op_b);
                                q.advance(1, 0, a.e_s);
                            }
                        }
                        pos.advance(step_s, step_x, a.e_s);
                    }
                }
                __syncthreads();
                for(uint32_t u = tid; u < nrv; u += NT)
                {
                    const uint32_t s = u / VPR, xv = u % VPR;
                    if(xv * VS < cnt)
                    {
                        Vec<T, VS> o;
#pragma unroll
                        for(int e = 0; e < VS; ++e)
                            o.v[e] = tile[s * PITCH + xv * VS + e];
                        store_stream<T, VS>(B + boff + xv * VS + s * a.row_stride, o);
                    }
                }
            }
        }

        struct QArgs
        {
            GroupShape  s;
            const void* A;
            void*       B;
            int32_t     bands, keep; // as in PArgs
            float       alpha;
            int32_t     op_a, op_b;
        };

        // Row x of a tile is (x0, x1) = (x mod w_i, x div w_i): x0 walks w_i elements of mode 0 and,
        // when the tile takes all of mode 0, x1 walks c_i indices of A's next mode - the two are
        // contiguous in A, so a row is one run of A.  Column y is (y0, y1) over mode j and B's next
        // mode in the same way, one run of B.  Rows are read along x, the tile is parked in LDS as
        // [y][x], and columns are written along y.
        // Narrow vectors are bound by the number of accesses, not by their bytes.  LOOSE: 16-byte vectors
        // whatever the extents; they start at any element, and the last one of a run is moved back to end with it
        // (its first elements are moved twice, to the same place).  Runs shorter than a vector, which only the
        // ragged tiles at the edges have, are moved by elements.
        // f16 21.25.23.57.25 -> (4,2,1,3,0), 34 MB: 43.4 -> 29.4 us; f16 129.513.65 -> (2,0,1) 14.2 -> 8.4; f32 21.25.23.57.25
        // 53.6 -> 43.0; f32 28.24.12.47.19.37 -> (4,2,3,0,5,1), 1 GB: 684 -> 634.
        template <typename T, int VR, int VW, bool LOOSE>
        __global__ __launch_bounds__(PERM_THREADS) void permute_group_kernel(QArgs a)
        {
            constexpr int NT = PERM_THREADS;
            constexpr int U  = 8;
            extern __shared__ unsigned char group_smem[];
            T* tile = reinterpret_cast<T*>(group_smem);

            const T* __restrict__ A = static_cast<const T*>(a.A);
            T* __restrict__ B       = static_cast<T*>(a.B);
            const uint32_t tid      = threadIdx.x;

            const GroupTile t     = group_tile(a.s, tile_work(blockIdx.x, gridDim.x, a.bands != 0));
            const uint32_t  RV    = group_per_line(a.s.w_i * a.s.c_i, VR, LOOSE), CV = group_per_line(a.s.w_j * a.s.c_j, VW, LOOSE);
            const T         alpha = static_cast<T>(a.alpha);

            auto read = [&](auto width, uint32_t per_row, uint32_t m_row) {
                constexpr int  W     = decltype(width)::value;
                const uint32_t total = per_row * t.ny;
                for(uint32_t u0 = 0; u0 < total; u0 += NT * U)
                {
                    Vec<T, W> r[U];
                    uint32_t  at[U];
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        const GroupVector g = group_read<W, LOOSE>(a.s, t, u0 + tid + k * NT, per_row, m_row);
                        at[k]               = g.ok ? g.line * a.s.pitch + g.at : 0xFFFFFFFFu;
                        // out-of-range lanes load the tile's first element: no branch, all loads in flight
                        const T* from = A + t.aoff + (g.ok ? g.at + g.off : 0u);
                        if constexpr(LOOSE && W > 1)
                            r[k] = load_loose(from);
                        else
                            r[k] = load_stream<T, W>(from);
                    }
#pragma unroll
                    for(int k = 0; k < U; ++k)
                    {
                        if(at[k] != 0xFFFFFFFFu)
                        {
#pragma unroll
                            for(int e = 0; e < W; ++e)
                                tile[at[k] + e] = element_op(r[k].v[e], alpha, a.op_a, a.op_b);
                        }
                    }
                }
            };
            auto write = [&](auto width, auto keep_c, uint32_t per_col, uint32_t m_col) {
                constexpr int  W     = decltype(width)::value;
                const uint32_t total = per_col * t.nx;
                for(uint32_t v = tid; v < total; v += NT)
                {
                    const GroupVector g = group_write<W, LOOSE>(a.s, t, v, per_col, m_col);
                    if(g.ok)
                    {
                        Vec<T, W> o;
#pragma unroll
                        for(int e = 0; e < W; ++e)
                            o.v[e] = tile[(g.at + e) * a.s.pitch + g.line];
                        T* to = B + t.boff + g.at + g.off;
                        if constexpr(decltype(keep_c)::value)
                            __builtin_memcpy(to, &o, sizeof(o));
                        else if constexpr(LOOSE && W > 1)
                            store_loose(to, o);
                        else
                            store_stream<T, W>(to, o);
                    }
                }
            };
            typedef std::integral_constant<int, 1> One;
            if(!LOOSE || t.nx >= VR)
                read(std::integral_constant<int, VR>{}, RV, a.s.m_rv);
            else
                read(One{}, group_singles(t.nx), recip(group_singles(t.nx)));
            __syncthreads();
            typedef std::integral_constant<bool, true> Keep;
            if(LOOSE && t.ny < VW)
                write(One{}, Keep{}, group_singles(t.ny), recip(group_singles(t.ny)));
            else if(a.keep)
                write(std::integral_constant<int, VW>{}, Keep{}, CV, a.s.m_cv);
            else
                write(std::integral_constant<int, VW>{}, std::integral_constant<bool, false>{}, CV, a.s.m_cv);
        }

        struct HArgs
        {
            const void* A;
            void*       B;
            uint32_t    e_c, e_i, e_j; // extents of mode 0, of A's next mode i and of B's next mode j
            uint32_t    c_i, c_j; // indices of i / j per tile
            uint32_t    a_j, b_i; // A stride of j, B stride of i (a_i == b_j == e_c)
            uint32_t    nt_i, nt_j;
            uint32_t    pitch; // LDS row pitch in elements: an odd number of 32-bit words
            uint32_t    m_rv, m_cv, m_ec; // floor(2^32 / d) + 1 for d = e_c * c_i / VR, e_c * c_j / VW, e_c
            int32_t     nb;
            uint32_t    bext[PERM_BATCH], ba[PERM_BATCH], bb[PERM_BATCH];
            float       alpha;
            int32_t     op_a, op_b;
        };

        // A and B share the fastest mode c.  The tile (c, i-chunk, j-chunk) is read as c_j runs of
        // e_c * c_i elements (c and i are contiguous in A), parked in LDS as [j][i * e_c + c], and
        // written as c_i runs of e_c * c_j elements (c and j are contiguous in B).
        template <typename T, int VR, int VW>
        __global__ __launch_bounds__(PERM_THREADS) void permute_shared_kernel(HArgs a)
        {
            constexpr int NT = PERM_THREADS;
            constexpr int U  = 8;
            extern __shared__ unsigned char shared_smem[];
            T* tile = reinterpret_cast<T*>(shared_smem);

            const T* __restrict__ A = static_cast<const T*>(a.A);
            T* __restrict__ B       = static_cast<T*>(a.B);
            const uint32_t tid      = threadIdx.x;

            uint32_t       blk = blockIdx.x;
            const uint32_t ti  = blk % a.nt_i;
            blk /= a.nt_i;
            const uint32_t tj = blk % a.nt_j;
            blk /= a.nt_j;
            uint32_t aoff = 0, boff = 0;
            for(int d = 0; d < a.nb; ++d)
            {
                const uint32_t c = blk % a.bext[d];
                blk /= a.bext[d];
                aoff += c * a.ba[d];
                boff += c * a.bb[d];
            }
            const uint32_t is = ti * a.c_i, js = tj * a.c_j;
            const uint32_t ci = (a.e_i - is) < a.c_i ? (a.e_i - is) : a.c_i;
            const uint32_t cj = (a.e_j - js) < a.c_j ? (a.e_j - js) : a.c_j;
            const uint32_t nx = a.e_c * ci, ny = a.e_c * cj; // run lengths inside the extents
            const uint32_t RV = a.e_c * a.c_i / VR, CV = a.e_c * a.c_j / VW; // vectors per nominal run
            aoff += is * a.e_c + js * a.a_j;
            boff += is * a.b_i + js * a.e_c;
            const T alpha = static_cast<T>(a.alpha);

            const uint32_t total_r = RV * cj;
            for(uint32_t u0 = 0; u0 < total_r; u0 += NT * U)
            {
                Vec<T, VR> r[U];
                uint32_t   at[U];
#pragma unroll
                for(int k = 0; k < U; ++k)
                {
                    const uint32_t v  = u0 + tid + k * NT;
                    const uint32_t y1 = __umulhi(v, a.m_rv), xv = v - y1 * RV;
                    const bool     ok = v < total_r && xv * VR < nx;
                    at[k]             = ok ? y1 * a.pitch + xv * VR : 0xFFFFFFFFu;
                    r[k] = load_stream<T, VR>(A + aoff + (ok ? xv * VR + y1 * a.a_j : 0u));
                }
#pragma unroll
                for(int k = 0; k < U; ++k)
                {
                    if(at[k] != 0xFFFFFFFFu)
                    {
#pragma unroll
                        for(int e = 0; e < VR; ++e)
                            tile[at[k] + e] = element_op(r[k].v[e], alpha, a.op_a, a.op_b);
                    }
                }
            }
            __syncthreads();
            const uint32_t total_w = CV * ci;
            for(uint32_t v = tid; v < total_w; v += NT)
            {
                const uint32_t x1 = __umulhi(v, a.m_cv), yv = v - x1 * CV;
                if(yv * VW < ny)
                {
                    const uint32_t y1 = __umulhi(yv * VW, a.m_ec), c = yv * VW - y1 * a.e_c;
                    Vec<T, VW>     o;
#pragma unroll
                    for(int e = 0; e < VW; ++e)
                        o.v[e] = tile[y1 * a.pitch + x1 * a.e_c + c + e];
                    store_stream<T, VW>(B + boff + yv * VW + x1 * a.b_i, o);
                }
            }
        }

        template <typename T, int V>
        __global__ __launch_bounds__(PERM_THREADS) void permute_copy_kernel(
            const void* Av, void* Bv, uint32_t nvec, float alphaF, int op_a, int op_b)
        {
            constexpr int U = 4;
            const auto*   A = static_cast<const Vec<T, V>*>(Av);
            auto*         B = static_cast<Vec<T, V>*>(Bv);
            const T       alpha = static_cast<T>(alphaF);
            const uint32_t base = blockIdx.x * (PERM_THREADS * U) + threadIdx.x;
            Vec<T, V>      r[U];
#pragma unroll
            for(int u = 0; u < U; ++u)
            {
                const uint32_t idx = base + u * PERM_THREADS;
                r[u]               = load_stream<T, V>(reinterpret_cast<const T*>(A + (idx < nvec ? idx : 0u)));
            }
#pragma unroll
            for(int u = 0; u < U; ++u)
            {
                const uint32_t idx = base + u * PERM_THREADS;
#pragma unroll
                for(int e = 0; e < V; ++e)
                    r[u].v[e] = element_op(r[u].v[e], alpha, op_a, op_b);
                if(idx < nvec)
                    store_stream<T, V>(reinterpret_cast<T*>(B + idx), r[u]);
            }
        }

        template <typename T>
        __global__ __launch_bounds__(PERM_THREADS) void permute_gather_kernel(GArgs g)
        {
            const uint32_t idx = blockIdx.x * PERM_THREADS + threadIdx.x;
            if(idx >= g.n)
                return;
            // index -> coordinates by multiplication: with m = floor(2^32 / e) + 1 the high word of
            // rem * m is the quotient or one more, for every 32-bit rem; one compare corrects it
            uint32_t rem = idx, aoff = 0;
            for(int d = 0; d < g.rank; ++d)
            {
                const uint32_t e = g.ext[d];
                uint32_t       q = __umulhi(rem, g.magic[d]);
                uint32_t       c = rem - q * e;
                if((int32_t)c < 0)
                {
                    q -= 1;
                    c += e;
                }
                rem = q;
                aoff += c * g.astr[d];
            }
            const T alpha               = static_cast<T>(g.alpha);
            static_cast<T*>(g.B)[idx] = element_op(static_cast<const T*>(g.A)[aoff], alpha, g.op_a, g.op_b);
        }

        struct RArgs
        {
            RunsShape   s;
            const void* A;
            void*       B;
            float       alpha;
            int32_t     op_a, op_b;
        };

        // A and B share the fastest mode, of V = 16 bytes' worth of elements or more.  Bound by HBM.  A tile of two modes
        // wastes the lanes that overhang them, and needs vectors that divide the run; here a vector is any V consecutive
        // elements of B, taken from A in one load at whatever address they have there (global memory takes 16-byte loads
        // and stores at any multiple of the element), or in two where the vector spans the end of a run.
        // f32 21.79.79.20.8.7 -> (0,1,3,4,5,2), 587 MB: 447 us in tiles, 198 here (5.9 TB/s); f32 30.7.61.7.7.65 ->
        // (0,4,2,3,1,5), 163 MB in runs of 120 bytes: 470 -> 81 us (4.0 TB/s: the run's ends share lines with others').
        // A thread moves U vectors, both loads of each in flight with the others'.
        template <typename T, int U>
        __global__ __launch_bounds__(PERM_THREADS) void permute_runs_kernel(RArgs a)
        {
            constexpr int V = 16 / (int)sizeof(T);
            typedef Vec<T, V> Elems;
            const T* __restrict__ A = static_cast<const T*>(a.A);
            T* __restrict__ B       = static_cast<T*>(a.B);
            const T alpha           = static_cast<T>(a.alpha);
            auto    load            = [&](uint32_t off) { return load_loose(A + off); };

            const uint32_t last  = a.s.n - V; // the last vector is moved back to end with the tensor
            const uint32_t first = (blockIdx.x * (PERM_THREADS * U) + threadIdx.x) * V;
            RunsVector     r[U];
            Elems          x[U], y[U];
#pragma unroll
            for(int u = 0; u < U; ++u)
            {
                const uint32_t at = first + u * PERM_THREADS * V;
                r[u]              = runs_vector(a.s, at < last ? at : last);
                x[u]              = load(r[u].src);
                if(r[u].left < V)
                    y[u] = load(r[u].next - r[u].left);
            }
#pragma unroll
            for(int u = 0; u < U; ++u)
            {
                const uint32_t k = r[u].left;
                if(k < V)
                {
#pragma unroll
                    for(int e = 1; e < V; ++e)
                        x[u].v[e] = (uint32_t)e < k ? x[u].v[e] : y[u].v[e];
                }
                const uint32_t at = first + u * PERM_THREADS * V;
#pragma unroll
                for(int e = 0; e < V; ++e)
                    x[u].v[e] = element_op(x[u].v[e], alpha, a.op_a, a.op_b);
                if(at < a.s.n)
                    store_loose(B + (at < last ? at : last), x[u]);
            }
        }

        // ---------------------------------------------------------------- host side

        struct TileShape
        {
            int ti, tj;
        };
        // element tiles per element size: square, long along i, long along j, and a 64 KiB tile
        // (512 threads, TILED only) whose rows and columns are twice as long as the square's
        constexpr int       NUM_TILES         = 4;
        constexpr TileShape TILES4[NUM_TILES] = {{64, 64}, {256, 16}, {16, 256}, {128, 128}};
        constexpr TileShape TILES2[NUM_TILES] = {{128, 128}, {512, 32}, {32, 512}, {256, 128}};

        template <typename T, int TI, int TJ, int VR, int VW, bool TR, bool BIG, bool LOOSE = false>
        int launch_tile(const PArgs& a, uint32_t grid, hipStream_t s)
        {
            if constexpr(BIG)
            {
                if constexpr(TR)
                    hipLaunchKernelGGL((permute_tile_kernel<T, TI, TJ, VR, VW, true, LOOSE, 512, true>), dim3(grid), dim3(512), 0, s, a);
                else
                    return -1;
            }
            else
                hipLaunchKernelGGL((permute_tile_kernel<T, TI, TJ, VR, VW, TR, LOOSE>), dim3(grid), dim3(PERM_THREADS), 0, s, a);
            return (int)hipGetLastError();
        }

        template <typename T, int TI, int TJ, int VMAX, bool BIG = false>
        int launch_tile_vec(bool transpose, bool loose, int vr, int vw, const PArgs& a, uint32_t grid, hipStream_t s)
        {
            if(loose)
                return launch_tile<T, TI, TJ, VMAX, VMAX, true, BIG, true>(a, grid, s);
#define HIPTK_PERM_CASE(R, W)                                                   \
    if(vr == R && vw == W)                                                      \
        return transpose ? launch_tile<T, TI, TJ, R, W, true, BIG>(a, grid, s)   \
                         : (R == W ? launch_tile<T, TI, TJ, R, R, false, BIG>(a, grid, s) : -1);
            HIPTK_PERM_CASE(1, 1)
            HIPTK_PERM_CASE(1, 2)
            HIPTK_PERM_CASE(1, VMAX)
            HIPTK_PERM_CASE(2, 1)
            HIPTK_PERM_CASE(2, 2)
            HIPTK_PERM_CASE(2, VMAX)
            HIPTK_PERM_CASE(VMAX, 1)
            HIPTK_PERM_CASE(VMAX, 2)
            HIPTK_PERM_CASE(VMAX, VMAX)
#undef HIPTK_PERM_CASE
            return -1;
        }

        template <typename T, int VMAX>
        int launch_tile_shape(int tile, bool transpose, bool loose, int vr, int vw, const PArgs& a, uint32_t grid, hipStream_t s)
        {
            constexpr const TileShape* TS = sizeof(T) == 4 ? TILES4 : TILES2;
            switch(tile)
            {
            case 0: return launch_tile_vec<T, TS[0].ti, TS[0].tj, VMAX>(transpose, loose, vr, vw, a, grid, s);
            case 1: return launch_tile_vec<T, TS[1].ti, TS[1].tj, VMAX>(transpose, loose, vr, vw, a, grid, s);
            case 2: return launch_tile_vec<T, TS[2].ti, TS[2].tj, VMAX>(transpose, loose, vr, vw, a, grid, s);
            case 3: return launch_tile_vec<T, TS[3].ti, TS[3].tj, VMAX, true>(transpose, loose, vr, vw, a, grid, s);
            default: return -1;
            }
        }

        template <typename T>
        int launch_copy(int vec, const void* A, void* B, uint32_t n, float alpha, int oa, int ob, hipStream_t s)
        {
            const uint32_t nvec = n / vec;
            const uint32_t grid = (nvec + PERM_THREADS * 4 - 1) / (PERM_THREADS * 4);
#define HIPTK_COPY_CASE(V)                                                                                           \
    if(vec == V)                                                                                                     \
    {                                                                                                                \
        hipLaunchKernelGGL((permute_copy_kernel<T, V>), dim3(grid), dim3(PERM_THREADS), 0, s, A, B, nvec, alpha, oa, ob); \
        return (int)hipGetLastError();                                                                               \
    }
            HIPTK_COPY_CASE(1)
            HIPTK_COPY_CASE(2)
            HIPTK_COPY_CASE(4)
            if constexpr(sizeof(T) == 2)
            {
                HIPTK_COPY_CASE(8)
            }
#undef HIPTK_COPY_CASE
            return -1;
        }

        // Strips hold e_s rows of TL elements in LDS (about 32 KiB at most): 2 KiB rows while the
        // short mode has at most 8 elements, 512-byte rows up to 64.
        constexpr int STRIP_MAX_SHORT = 64;
        constexpr int STRIP_WIDE_MAX  = 8;

        constexpr int strip_len(int elem_bytes, int e_s)
        {
            return (e_s <= STRIP_WIDE_MAX ? 2048 : 512) / elem_bytes;
        }

        template <typename T, int VMAX, int TL>
        int launch_strip_len(bool linear_write, int vl, int vs, const SArgs& a, uint32_t grid, hipStream_t s)
        {
            const size_t lds = (size_t)a.e_s * (TL * sizeof(T) + 4);
#define HIPTK_STRIP_CASE(L, S)                                                                                      \
    if(vl == L && vs == S)                                                                                          \
    {                                                                                                               \
        if(linear_write)                                                                                            \
            hipLaunchKernelGGL((permute_strip_kernel<T, TL, L, S, true>), dim3(grid), dim3(PERM_THREADS), lds, s, a);  \
        else                                                                                                        \
            hipLaunchKernelGGL((permute_strip_kernel<T, TL, L, S, false>), dim3(grid), dim3(PERM_THREADS), lds, s, a); \
        return (int)hipGetLastError();                                                                              \
    }
            HIPTK_STRIP_CASE(1, 1)
            HIPTK_STRIP_CASE(1, 2)
            HIPTK_STRIP_CASE(1, VMAX)
            HIPTK_STRIP_CASE(2, 1)
            HIPTK_STRIP_CASE(2, 2)
            HIPTK_STRIP_CASE(2, VMAX)
            HIPTK_STRIP_CASE(VMAX, 1)
            HIPTK_STRIP_CASE(VMAX, 2)
            HIPTK_STRIP_CASE(VMAX, VMAX)
#undef HIPTK_STRIP_CASE
            return -1;
        }

        template <typename T, int VMAX>
        int launch_strip(bool linear_write, int vl, int vs, const SArgs& a, uint32_t grid, hipStream_t s)
        {
            if(a.e_s <= (uint32_t)STRIP_WIDE_MAX)
                return launch_strip_len<T, VMAX, strip_len(sizeof(T), 1)>(linear_write, vl, vs, a, grid, s);
            return launch_strip_len<T, VMAX, strip_len(sizeof(T), STRIP_MAX_SHORT)>(linear_write, vl, vs, a, grid, s);
        }

        constexpr int GROUP_MAX_FAST = 128; // longest fastest mode the grouped kernel takes
        constexpr int GROUP_MAX_LDS  = 60 * 1024;

        template <typename T, int VMAX>
        int launch_group(int vr, int vw, bool loose, const QArgs& a, uint32_t grid, size_t lds, hipStream_t s)
        {
            if(loose)
            {
                hipLaunchKernelGGL((permute_group_kernel<T, VMAX, VMAX, true>), dim3(grid), dim3(PERM_THREADS), lds, s, a);
                return (int)hipGetLastError();
            }
#define HIPTK_GROUP_CASE(R, W)                                                                                     \
    if(vr == R && vw == W)                                                                                         \
    {                                                                                                              \
        hipLaunchKernelGGL((permute_group_kernel<T, R, W, false>), dim3(grid), dim3(PERM_THREADS), lds, s, a);              \
        return (int)hipGetLastError();                                                                             \
    }
            HIPTK_GROUP_CASE(1, 1)
            HIPTK_GROUP_CASE(1, 2)
            HIPTK_GROUP_CASE(1, VMAX)
            HIPTK_GROUP_CASE(2, 1)
            HIPTK_GROUP_CASE(2, 2)
            HIPTK_GROUP_CASE(2, VMAX)
            HIPTK_GROUP_CASE(VMAX, 1)
            HIPTK_GROUP_CASE(VMAX, 2)
            HIPTK_GROUP_CASE(VMAX, VMAX)
#undef HIPTK_GROUP_CASE
            return -1;
        }

        template <typename T, int VMAX>
        int launch_shared(int v, const HArgs& a, uint32_t grid, size_t lds, hipStream_t s)
        {
#define HIPTK_SHARED_CASE(V)                                                                                  \
    if(v == V)                                                                                                \
    {                                                                                                         \
        hipLaunchKernelGGL((permute_shared_kernel<T, V, V>), dim3(grid), dim3(PERM_THREADS), lds, s, a);        \
        return (int)hipGetLastError();                                                                        \
    }
            HIPTK_SHARED_CASE(1)
            HIPTK_SHARED_CASE(2)
            HIPTK_SHARED_CASE(VMAX)
#undef HIPTK_SHARED_CASE
            return -1;
        }

        bool vec_allowed(int elem_bytes, int v)
        {
            return v == 1 || v == 2 || (elem_bytes == 4 ? v == 4 : v == 8);
        }
        bool copy_vec_allowed(int elem_bytes, int v)
        {
            return v == 1 || v == 2 || v == 4 || (elem_bytes == 2 && v == 8);
        }

        bool aligned(const void* p, int bytes)
        {
            return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)bytes) == 0;
        }

        // Shape checks shared by the name query and the launcher.
        bool well_formed(const hiptk_permute_t* p, int64_t* count)
        {
            if(!p || (p->elem_bytes != 2 && p->elem_bytes != 4) || p->rank < 1 || p->rank > HIPTK_PERM_MAX_RANK)
                return false;
            if(((p->op_a | p->op_b) & ~1) && !(p->op_a == HIPTK_PERM_OP_RAW && p->op_b == 0))
                return false;
            int64_t n = 1;
            for(int d = 0; d < p->rank; ++d)
            {
                if(p->extent[d] < 1 || p->a_stride[d] < 1 || p->b_stride[d] < 1)
                    return false;
                n *= p->extent[d];
                if(n >= (int64_t(1) << 31))
                    return false;
            }
            // A is packed in the order given
            int64_t s = 1;
            for(int d = 0; d < p->rank; ++d)
            {
                if(p->a_stride[d] != s)
                    return false;
                s *= p->extent[d];
            }
            // B is packed in some order of the same modes
            int order[HIPTK_PERM_MAX_RANK];
            for(int d = 0; d < p->rank; ++d)
                order[d] = d;
            std::sort(order, order + p->rank, [p](int x, int y) {
                return p->b_stride[x] != p->b_stride[y] ? p->b_stride[x] < p->b_stride[y] : x < y;
            });
            s = 1;
            for(int d = 0; d < p->rank; ++d)
            {
                if(p->b_stride[order[d]] != s)
                    return false;
                s *= p->extent[order[d]];
            }
            *count = n;
            return true;
        }

        const char* type_tag(int elem_bytes)
        {
            return elem_bytes == 4 ? "f32" : "f16";
        }
    }
}

extern "C" const char* hiptk_permute_kernel_name(const hiptk_permute_t* p)
{
    using namespace hiptk;
    static thread_local char name[96];
    name[0]   = 0;
    int64_t n = 0;
    if(!well_formed(p, &n))
        return name;
    switch(p->kernel)
    {
    case HIPTK_PERM_COPY:
        if(p->rank == 1 && copy_vec_allowed(p->elem_bytes, p->vec_r))
            snprintf(name, sizeof(name), "permute_copy_%s_v%d", type_tag(p->elem_bytes), p->vec_r);
        break;
    case HIPTK_PERM_TILED:
    case HIPTK_PERM_ROWS:
    {
        if(p->tile < 0 || p->tile >= NUM_TILES || !vec_allowed(p->elem_bytes, p->vec_r) || !vec_allowed(p->elem_bytes, p->vec_w))
            break;
        if(p->kernel == HIPTK_PERM_ROWS && (p->vec_r != p->vec_w || p->tile == 3))
            break;
        const TileShape t = (p->elem_bytes == 4 ? TILES4 : TILES2)[p->tile];
        snprintf(name,
                 sizeof(name),
                 p->kernel == HIPTK_PERM_TILED && p->loose ? "permute_%s_%s_%dx%d_r%d_w%d_loose" : "permute_%s_%s_%dx%d_r%d_w%d",
                 p->kernel == HIPTK_PERM_TILED ? "tiled" : "rows",
                 type_tag(p->elem_bytes),
                 t.ti,
                 t.tj,
                 p->vec_r,
                 p->vec_w);
        break;
    }
    case HIPTK_PERM_GATHER: snprintf(name, sizeof(name), "permute_gather_%s", type_tag(p->elem_bytes)); break;
    case HIPTK_PERM_RUNS:
        if(p->vec_r * p->elem_bytes == 16 && p->vec_w == p->vec_r)
            snprintf(name, sizeof(name), "permute_runs_%s_%d_v%dx%d", type_tag(p->elem_bytes), p->extent[0], p->vec_r, runs_per_thread(n, p->vec_r));
        break;
    case HIPTK_PERM_GROUPED:
        if(vec_allowed(p->elem_bytes, p->vec_r) && vec_allowed(p->elem_bytes, p->vec_w) && p->chunk_i >= 1 && p->chunk_j >= 1)
            snprintf(name,
                     sizeof(name),
                     p->loose ? "permute_grouped_%s_%dx%d_r%d_w%d_loose" : "permute_grouped_%s_%dx%d_r%d_w%d",
                     type_tag(p->elem_bytes),
                     p->width_i * p->chunk_i,
                     p->width_j * p->chunk_j,
                     p->vec_r,
                     p->vec_w);
        break;
    case HIPTK_PERM_SHARED:
        if(vec_allowed(p->elem_bytes, p->vec_r) && p->vec_r == p->vec_w && p->chunk_i >= 1 && p->chunk_j >= 1)
            snprintf(name,
                     sizeof(name),
                     "permute_shared_%s_%dx%dx%d_v%d",
                     type_tag(p->elem_bytes),
                     p->extent[0],
                     p->chunk_i,
                     p->chunk_j,
                     p->vec_r);
        break;
    case HIPTK_PERM_STRIP:
        if((p->tile == 0 || p->tile == 1) && p->mode_j >= 1 && p->mode_j < p->rank && vec_allowed(p->elem_bytes, p->vec_r)
           && vec_allowed(p->elem_bytes, p->vec_w))
            snprintf(name,
                     sizeof(name),
                     "permute_strip_%s_%s_%d_r%d_w%d",
                     type_tag(p->elem_bytes),
                     p->tile == 0 ? "linear_write" : "linear_read",
                     strip_len(p->elem_bytes, p->extent[p->tile == 0 ? p->mode_j : 0]),
                     p->vec_r,
                     p->vec_w);
        break;
    default: break;
    }
    return name;
}

extern "C" int hiptk_permute(const hiptk_permute_t* p, const void* A, void* B, void* stream, int* hip_error)
{
    using namespace hiptk;
    if(hip_error)
        *hip_error = 0;
    int64_t n = 0;
    if(!well_formed(p, &n) || !A || !B)
        return HIPTK_ERR_ARG;
    if(!aligned(A, p->elem_bytes) || !aligned(B, p->elem_bytes) || (p->a_align > 1 && !aligned(A, p->a_align)))
        return HIPTK_ERR_ARG;
    hipStream_t s  = static_cast<hipStream_t>(stream);
    int         rc = -1;

    if(p->kernel == HIPTK_PERM_COPY)
    {
        const int v = p->vec_r;
        if(p->rank != 1 || !copy_vec_allowed(p->elem_bytes, v))
            return HIPTK_ERR_NO_KERNEL;
        if(n % v != 0 || !aligned(A, v * p->elem_bytes) || !aligned(B, v * p->elem_bytes))
            return HIPTK_ERR_ARG;
        rc = p->elem_bytes == 4 ? launch_copy<float>(v, A, B, (uint32_t)n, p->alpha, p->op_a, p->op_b, s)
                                : launch_copy<_Float16>(v, A, B, (uint32_t)n, p->alpha, p->op_a, p->op_b, s);
    }
    else if(p->kernel == HIPTK_PERM_GATHER)
    {
        GArgs g;
        memset(&g, 0, sizeof(g));
        g.A     = A;
        g.B     = B;
        g.n     = (uint32_t)n;
        g.rank  = p->rank;
        g.alpha = p->alpha;
        g.op_a  = p->op_a;
        g.op_b  = p->op_b;
        int order[HIPTK_PERM_MAX_RANK];
        for(int d = 0; d < p->rank; ++d)
            order[d] = d;
        std::sort(order, order + p->rank, [p](int x, int y) {
            return p->b_stride[x] != p->b_stride[y] ? p->b_stride[x] < p->b_stride[y] : x < y;
        });
        int kept = 0;
        for(int d = 0; d < p->rank; ++d)
        {
            const uint32_t e = (uint32_t)p->extent[order[d]];
            if(e == 1)
                continue; // its coordinate is always 0
            g.ext[kept]   = e;
            g.astr[kept]  = (uint32_t)p->a_stride[order[d]];
            g.magic[kept] = magic_of(e);
            ++kept;
        }
        g.rank = kept;
        const uint32_t grid = (uint32_t)((n + PERM_THREADS - 1) / PERM_THREADS);
        if(p->elem_bytes == 4)
            hipLaunchKernelGGL((permute_gather_kernel<float>), dim3(grid), dim3(PERM_THREADS), 0, s, g);
        else
            hipLaunchKernelGGL((permute_gather_kernel<_Float16>), dim3(grid), dim3(PERM_THREADS), 0, s, g);
        rc = (int)hipGetLastError();
    }
    else if(p->kernel == HIPTK_PERM_RUNS)
    {
        const int v = 16 / p->elem_bytes;
        if(p->vec_r != v || p->vec_w != v)
            return HIPTK_ERR_NO_KERNEL;
        // one run at least in every vector's reach, so that a vector spans two at the most; the reciprocals want
        // divisors of 2 and more
        if(p->rank < 2 || p->b_stride[0] != 1 || p->extent[0] < v)
            return HIPTK_ERR_ARG;
        RArgs a;
        memset(&a, 0, sizeof(a));
        a.A     = A;
        a.B     = B;
        a.s     = runs_shape(*p, n);
        a.alpha = p->alpha;
        a.op_a  = p->op_a;
        a.op_b  = p->op_b;
        const int      u    = runs_per_thread(n, v);
        const int64_t  per  = (int64_t)PERM_THREADS * u * v;
        const uint32_t grid = (uint32_t)((n + per - 1) / per);
        if(p->elem_bytes == 4 && u == 4)
            hipLaunchKernelGGL((permute_runs_kernel<float, 4>), dim3(grid), dim3(PERM_THREADS), 0, s, a);
        else if(p->elem_bytes == 4)
            hipLaunchKernelGGL((permute_runs_kernel<float, 1>), dim3(grid), dim3(PERM_THREADS), 0, s, a);
        else if(u == 4)
            hipLaunchKernelGGL((permute_runs_kernel<_Float16, 4>), dim3(grid), dim3(PERM_THREADS), 0, s, a);
        else
            hipLaunchKernelGGL((permute_runs_kernel<_Float16, 1>), dim3(grid), dim3(PERM_THREADS), 0, s, a);
        rc = (int)hipGetLastError();
    }
    else if(p->kernel == HIPTK_PERM_TILED || p->kernel == HIPTK_PERM_ROWS)
    {
        const bool transpose = p->kernel == HIPTK_PERM_TILED;
        const int  mi = p->mode_i, mj = p->mode_j;
        if(p->rank < 2 || mi != 0 || mj < 1 || mj >= p->rank || p->tile < 0 || p->tile >= NUM_TILES)
            return HIPTK_ERR_ARG;
        if(!vec_allowed(p->elem_bytes, p->vec_r) || !vec_allowed(p->elem_bytes, p->vec_w))
            return HIPTK_ERR_NO_KERNEL;
        if(!transpose && p->vec_r != p->vec_w)
            return HIPTK_ERR_NO_KERNEL;
        // the layout each kernel assumes
        if(transpose ? p->b_stride[mj] != 1 : p->b_stride[0] != 1)
            return HIPTK_ERR_ARG;
        // what the vector widths assume: whole vectors inside the extents, every other
        // stride and both base pointers multiples of the vector
        // (loose: 16 bytes at any element)
        const int  vr = p->vec_r, vw = p->vec_w;
        const bool loose = transpose && p->loose != 0;
        const int  wmode = transpose ? mj : 0; // the mode stores run along
        if(loose && (vr * p->elem_bytes != 16 || vw != vr))
            return HIPTK_ERR_ARG;
        if(!loose)
        {
            if(p->extent[0] % vr != 0 || !aligned(A, vr * p->elem_bytes))
                return HIPTK_ERR_ARG;
            for(int d = 1; d < p->rank; ++d)
                if(p->a_stride[d] % vr != 0)
                    return HIPTK_ERR_ARG;
            if(p->extent[wmode] % vw != 0 || !aligned(B, vw * p->elem_bytes))
                return HIPTK_ERR_ARG;
            for(int d = 0; d < p->rank; ++d)
                if(d != wmode && p->b_stride[d] % vw != 0)
                    return HIPTK_ERR_ARG;
        }

        const TileShape t = (p->elem_bytes == 4 ? TILES4 : TILES2)[p->tile];
        PArgs           a;
        memset(&a, 0, sizeof(a));
        a.A     = A;
        a.B     = B;
        a.e_i   = (uint32_t)p->extent[0];
        a.e_j   = (uint32_t)p->extent[mj];
        a.a_j   = (uint32_t)p->a_stride[mj];
        a.b_i   = (uint32_t)p->b_stride[0];
        a.b_j   = (uint32_t)p->b_stride[mj];
        a.nt_i  = (a.e_i + t.ti - 1) / t.ti;
        a.nt_j  = (a.e_j + t.tj - 1) / t.tj;
        a.group = p->group == 0 ? 0u : (uint32_t)std::max(1, std::min(p->group, (int32_t)a.nt_j));
        a.bands = p->bands != 0;
        a.keep  = p->keep != 0;
        a.alpha = p->alpha;
        a.op_a  = p->op_a;
        a.op_b  = p->op_b;
        int64_t grid = (int64_t)a.nt_i * a.nt_j;
        for(int d = 1; d < p->rank; ++d)
        {
            if(d == mj)
                continue;
            a.bext[a.nb] = (uint32_t)p->extent[d];
            a.ba[a.nb]   = (uint32_t)p->a_stride[d];
            a.bb[a.nb]   = (uint32_t)p->b_stride[d];
            ++a.nb;
            grid *= p->extent[d];
        }
        if(grid >= (int64_t(1) << 31))
            return HIPTK_ERR_ARG;
        rc = p->elem_bytes == 4 ? launch_tile_shape<float, 4>(p->tile, transpose, loose, vr, vw, a, (uint32_t)grid, s)
                                : launch_tile_shape<_Float16, 8>(p->tile, transpose, loose, vr, vw, a, (uint32_t)grid, s);
    }
    else if(p->kernel == HIPTK_PERM_GROUPED)
    {
        const int mj = p->mode_j, mi2 = p->mode_i2, mj2 = p->mode_j2;
        if(p->rank < 2 || p->mode_i != 0 || mj < 1 || mj >= p->rank || p->b_stride[mj] != 1)
            return HIPTK_ERR_ARG;
        if(!vec_allowed(p->elem_bytes, p->vec_r) || !vec_allowed(p->elem_bytes, p->vec_w))
            return HIPTK_ERR_NO_KERNEL;
        // the second modes, where present, directly follow the first ones in memory and are
        // distinct from every other tile mode
        if(mi2 != -1 && (mi2 < 1 || mi2 >= p->rank || mi2 == mj || mi2 == mj2 || p->a_stride[mi2] != p->extent[0]))
            return HIPTK_ERR_ARG;
        if(mj2 != -1 && (mj2 < 1 || mj2 >= p->rank || mj2 == mj || p->b_stride[mj2] != p->extent[mj]))
            return HIPTK_ERR_ARG;
        const int e_i1 = mi2 == -1 ? 1 : p->extent[mi2], e_j1 = mj2 == -1 ? 1 : p->extent[mj2];
        const int w_i = p->width_i, w_j = p->width_j;
        if(w_i < 1 || w_i > p->extent[0] || w_j < 1 || w_j > p->extent[mj] || p->chunk_i < 1 || p->chunk_j < 1
           || p->chunk_i > e_i1 || p->chunk_j > e_j1)
            return HIPTK_ERR_ARG;
        // a tile takes several indices of a second mode only together with the whole first mode
        if((p->chunk_i > 1 && w_i != p->extent[0]) || (p->chunk_j > 1 && w_j != p->extent[mj]))
            return HIPTK_ERR_ARG;
        // vectors: whole vectors inside the tile widths and the fastest modes, every other stride
        // and both bases aligned
        // (loose: 16 bytes at any element)
        const int  vr = p->vec_r, vw = p->vec_w;
        const bool loose = p->loose != 0;
        if(loose && (vr * p->elem_bytes != 16 || vw != vr))
            return HIPTK_ERR_ARG;
        if(!loose)
        {
            if(p->extent[0] % vr != 0 || p->extent[mj] % vw != 0 || w_i % vr != 0 || w_j % vw != 0
               || !aligned(A, vr * p->elem_bytes) || !aligned(B, vw * p->elem_bytes))
                return HIPTK_ERR_ARG;
            for(int d = 1; d < p->rank; ++d)
                if(p->a_stride[d] % vr != 0)
                    return HIPTK_ERR_ARG;
            for(int d = 0; d < p->rank; ++d)
                if(d != mj && p->b_stride[d] % vw != 0)
                    return HIPTK_ERR_ARG;
        }

        QArgs a;
        memset(&a, 0, sizeof(a));
        a.A    = A;
        a.B    = B;
        const uint32_t TI = (uint32_t)w_i * (uint32_t)p->chunk_i, TJ = (uint32_t)w_j * (uint32_t)p->chunk_j;
        if(TI / vr < 2 || TJ / vw < 2 || w_i < 2 || w_j < 2)
            return HIPTK_ERR_ARG; // (the reciprocals are exact for divisors of 2 and more)
        int64_t grid = 0;
        a.s          = group_shape(*p, grid);
        a.bands      = p->bands != 0;
        a.keep       = p->keep != 0;
        a.alpha      = p->alpha;
        a.op_a       = p->op_a;
        a.op_b       = p->op_b;
        const size_t lds = (size_t)TJ * a.s.pitch * p->elem_bytes;
        if(lds > (size_t)GROUP_MAX_LDS || grid >= (int64_t(1) << 31))
            return HIPTK_ERR_ARG;
        rc = p->elem_bytes == 4 ? launch_group<float, 4>(vr, vw, loose, a, (uint32_t)grid, lds, s)
                                : launch_group<_Float16, 8>(vr, vw, loose, a, (uint32_t)grid, lds, s);
    }
    else if(p->kernel == HIPTK_PERM_SHARED)
    {
        const int mi = p->mode_i2, mj = p->mode_j2, v = p->vec_r;
        if(p->rank < 3 || p->mode_i != 0 || p->b_stride[0] != 1 || mi < 1 || mi >= p->rank || mj < 1 || mj >= p->rank || mi == mj)
            return HIPTK_ERR_ARG;
        if(p->a_stride[mi] != p->extent[0] || p->b_stride[mj] != p->extent[0])
            return HIPTK_ERR_ARG;
        if(!vec_allowed(p->elem_bytes, v) || p->vec_w != v)
            return HIPTK_ERR_NO_KERNEL;
        if(p->extent[0] > GROUP_MAX_FAST || p->chunk_i < 1 || p->chunk_j < 1 || p->chunk_i > p->extent[mi] || p->chunk_j > p->extent[mj])
            return HIPTK_ERR_ARG;
        if(p->extent[0] % v != 0 || !aligned(A, v * p->elem_bytes) || !aligned(B, v * p->elem_bytes))
            return HIPTK_ERR_ARG;
        for(int d = 1; d < p->rank; ++d)
            if(p->a_stride[d] % v != 0 || p->b_stride[d] % v != 0)
                return HIPTK_ERR_ARG;
        HArgs a;
        memset(&a, 0, sizeof(a));
        a.A    = A;
        a.B    = B;
        a.e_c  = (uint32_t)p->extent[0];
        a.e_i  = (uint32_t)p->extent[mi];
        a.e_j  = (uint32_t)p->extent[mj];
        a.c_i  = (uint32_t)p->chunk_i;
        a.c_j  = (uint32_t)p->chunk_j;
        a.a_j  = (uint32_t)p->a_stride[mj];
        a.b_i  = (uint32_t)p->b_stride[mi];
        a.nt_i = (a.e_i + a.c_i - 1) / a.c_i;
        a.nt_j = (a.e_j + a.c_j - 1) / a.c_j;
        const uint32_t TI = a.e_c * a.c_i, TJ = a.e_c * a.c_j;
        const uint32_t wordElems  = 4u / (uint32_t)p->elem_bytes;
        uint32_t       pitchWords = (TI + wordElems - 1) / wordElems;
        pitchWords |= 1u;
        a.pitch          = pitchWords * wordElems;
        const size_t lds = (size_t)a.c_j * a.pitch * p->elem_bytes;
        if(lds > (size_t)GROUP_MAX_LDS || TI / v < 2 || TJ / v < 2)
            return HIPTK_ERR_ARG;
        a.m_rv  = magic_of(TI / v);
        a.m_cv  = magic_of(TJ / v);
        a.m_ec  = magic_of(a.e_c);
        a.alpha = p->alpha;
        a.op_a  = p->op_a;
        a.op_b  = p->op_b;
        int64_t grid = (int64_t)a.nt_i * a.nt_j;
        for(int d = 1; d < p->rank; ++d)
        {
            if(d == mi || d == mj)
                continue;
            a.bext[a.nb] = (uint32_t)p->extent[d];
            a.ba[a.nb]   = (uint32_t)p->a_stride[d];
            a.bb[a.nb]   = (uint32_t)p->b_stride[d];
            ++a.nb;
            grid *= p->extent[d];
        }
        if(grid >= (int64_t(1) << 31))
            return HIPTK_ERR_ARG;
        rc = p->elem_bytes == 4 ? launch_shared<float, 4>(v, a, (uint32_t)grid, lds, s)
                                : launch_shared<_Float16, 8>(v, a, (uint32_t)grid, lds, s);
    }
    else if(p->kernel == HIPTK_PERM_STRIP)
    {
        // tile == 0: long mode 0 (A's fastest), short mode mode_j (B's fastest), B holds mode 0
        //            right after it; the strip is linear in B.
        // tile == 1: short mode 0 (A's fastest) with long mode mode_j right after it in A and
        //            fastest in B; the strip is linear in A.
        const int  mj           = p->mode_j;
        const bool linear_write = p->tile == 0;
        if(p->rank < 2 || p->mode_i != 0 || mj < 1 || mj >= p->rank || (p->tile != 0 && p->tile != 1))
            return HIPTK_ERR_ARG;
        if(!vec_allowed(p->elem_bytes, p->vec_r) || !vec_allowed(p->elem_bytes, p->vec_w))
            return HIPTK_ERR_NO_KERNEL;
        const int ms = linear_write ? mj : 0, ml = linear_write ? 0 : mj; // short, long
        if(p->extent[ms] > STRIP_MAX_SHORT || p->b_stride[mj] != 1)
            return HIPTK_ERR_ARG;
        if(linear_write ? p->b_stride[0] != p->extent[mj] : p->a_stride[mj] != p->extent[0])
            return HIPTK_ERR_ARG;
        // vector preconditions: the linear side needs whole vectors in every strip and aligned
        // strip starts, the row side whole vectors in every row
        const int     vr = p->vec_r, vw = p->vec_w;
        const int     vl = linear_write ? vw : vr, vs = linear_write ? vr : vw;
        const int64_t run = (int64_t)p->extent[0] * p->extent[mj];
        const int32_t* lin_stride = linear_write ? p->b_stride : p->a_stride;
        const int32_t* row_stride = linear_write ? p->a_stride : p->b_stride;
        if(run % vl != 0 || p->extent[ml] % vs != 0)
            return HIPTK_ERR_ARG;
        for(int d = 1; d < p->rank; ++d)
        {
            if(d != mj && lin_stride[d] % vl != 0)
                return HIPTK_ERR_ARG;
            if((d != mj || linear_write) && row_stride[d] % vs != 0)
                return HIPTK_ERR_ARG;
        }
        if(!linear_write && p->b_stride[0] % vs != 0)
            return HIPTK_ERR_ARG;
        if(!aligned(A, vr * p->elem_bytes) || !aligned(B, vw * p->elem_bytes))
            return HIPTK_ERR_ARG;

        const int TL = strip_len(p->elem_bytes, p->extent[ms]);
        SArgs     a;
        memset(&a, 0, sizeof(a));
        a.A          = A;
        a.B          = B;
        a.e_s        = (uint32_t)p->extent[ms];
        a.e_l        = (uint32_t)p->extent[ml];
        a.row_stride = (uint32_t)(linear_write ? p->a_stride[mj] : p->b_stride[0]);
        a.magic      = (uint32_t)((uint64_t(1) << 32) / a.e_s) + 1u;
        a.nt         = (a.e_l + TL - 1) / TL;
        a.alpha      = p->alpha;
        a.op_a       = p->op_a;
        a.op_b       = p->op_b;
        int64_t grid = a.nt;
        for(int d = 1; d < p->rank; ++d)
        {
            if(d == mj)
                continue;
            a.bext[a.nb] = (uint32_t)p->extent[d];
            a.ba[a.nb]   = (uint32_t)p->a_stride[d];
            a.bb[a.nb]   = (uint32_t)p->b_stride[d];
            ++a.nb;
            grid *= p->extent[d];
        }
        if(grid >= (int64_t(1) << 31))
            return HIPTK_ERR_ARG;
        rc = p->elem_bytes == 4 ? launch_strip<float, 4>(linear_write, vl, vs, a, (uint32_t)grid, s)
                                : launch_strip<_Float16, 8>(linear_write, vl, vs, a, (uint32_t)grid, s);
    }
    else
        return HIPTK_ERR_NO_KERNEL;

    if(rc == -1)
        return HIPTK_ERR_NO_KERNEL;
    if(hip_error)
        *hip_error = rc;
    return rc == 0 ? HIPTK_OK : HIPTK_ERR_LAUNCH;
}
