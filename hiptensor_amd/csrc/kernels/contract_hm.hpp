// 16-bit (f16 / bf16) contraction kernel for gfx950 with tiles of 64 and 128 rows and columns whose operand tiles go
// from global memory straight into LDS (global_load_lds_dwordx4), on v_mfma_f32_16x16x32.
//
// For outputs that 256-wide tiles (contract_hk.hpp, contract_hr.hpp) leave most compute units without work for.  Staged through
// registers (contract_h.hpp) a K step of 64 of a 64 x 64 tile took about 900 cycles there, the latency of its loads, for
// 128 cycles of MFMAs.  Here a ring of NS stages keeps up to NS K tiles on their way, two workgroups share a compute unit, and a
// step takes what the LDS takes for it: the loads written at 64 bytes a clock, the operands read at 232 (ds_read_b128) or
// 115 (transposing) - 64 x 64: 400 / 540 cycles, 350-390 / 510 measured (0.15 / 0.21 us); 128 x 64: 600 / 810, 620 / 870.
// 2048 x 512 x 1480 f16, both k-contiguous 13.9 -> 10.1 us; 1600 x 768 x 2012, both row-contiguous 19.1 -> 15.1;
// 1024 x 2048 x 768 bf16 9.7 -> 7.6; 11760 x 4 x 4112 f16 22.4 -> 20.9; 160 x 768 x 1152 bf16 8.7 (in four slices) -> 6.1.
// (Ring of 3 or 5 stages for 64 x 64: 0.95-1.10 of the time of 4; ring of 2 for 128 x 64: 1.0-1.5 of 3; tiles of 128 x 128 win
// on three of 62 drawn problems, by up to 12 %, and tiles of 32 rows on five, by 1-3 %: not built.)
//
//   * 256 threads, wave grid 2 x 2.  Stages, swizzles and operand fetches are those of contract_hk.hpp
//     (k-contiguous operand: stage[row][64], ds_read_b128; row-contiguous: stage[64][rows], ds_read_b64_tr_b16).
//   * A wave holds the operands of two K tiles in registers, as in contract_wd.hpp: behind the step's one barrier, which says
//     that every wave has tile t in registers and that tile t + 1 has landed, tile t + 1 is read from LDS, tile t + NS is
//     requested into the stage of tile t, and tile t is multiplied.  (Operands read in the step that multiplies them, so that a
//     wave alone on its SIMD waits for them: 2048 x 512 x 1480 12.4 us.)  The compiler orders the rest: the loads are
//     inline assembly, so its own wait counts leave them alone.
//   * Vectors may start at any 4 bytes (a direct load needs no more; 128-byte runs of a K tile then lie in two lines each and
//     come at half the rate).  Operands whose vectors start at odd elements are not offered.
//   * K tail: the tile that K ends in is taken first.  Vectors beyond K come from 16 bytes of zeros, so the tile multiplies as
//     a whole one and no address leaves the tensor.  Where K ends inside a vector of a k-contiguous operand, the vector is
//     loaded so that it ends with K, the other operand's k likewise, and the k it shares with the vector in front of it
//     are zeroed in the operand registers of both.
//   * Tiles that overhang P or Q read row 0 there (the tables' padding), or are moved back (shift_p / shift_q).
#pragma once
#include "contract_h.hpp"
#include "dma_lds.hpp"
#include "hd_addr.hpp"

namespace hiptk
{
    template <int BP_, int BQ_, int NS_>
    struct HmGeom
    {
        static constexpr int BP = BP_, BQ = BQ_, BK = HK_BK, NS = NS_;
        static constexpr int WP = 2, WQ = 2; // wave grid
        static constexpr int TP = BP / WP / 32, TQ = BQ / WQ / 32; // 32 x 32 blocks of a wave tile
        static constexpr int OPX = BP * BK, OPY = BQ * BK; // elements of an operand in one stage
        static constexpr int NXL = BP / 32, NYL = BQ / 32; // direct loads (1 KiB) per wave and K tile
        static constexpr int LPT = NXL + NYL;
        static constexpr int STAGE     = OPX + OPY;
        static constexpr int LDS_BYTES = NS * STAGE * 2;
        static_assert(TP >= 1 && TQ >= 1 && BP % (WP * 32) == 0 && BQ % (WQ * 32) == 0, "whole wave tiles");
        static_assert(NS >= 2 && (NS - 2) * LPT < 64, "the wait counts must fit vmcnt");
        static_assert(NS <= 4, "last_steps tells up to two tiles on their way apart");
        static_assert(LDS_BYTES <= 160 * 1024 && LDS_BYTES >= 4 * 32 * (TQ * 32 + 4) * 4, "LDS of one CU; the epilogue's staging");
    };

    // what the parts of the last K tile that lie beyond K are loaded from
    static __device__ __attribute__((aligned(16))) const unsigned char hm_zero16[16] = {0};

    // 2 or 4 direct loads into consecutive KiB of LDS from m0 on, in one statement: one write of M0 and one run of
    // wait states (see dma_lds.hpp) for all of them.  The offset field moves source and destination alike: the lanes' offsets
    // are lowered by as much (voff[i] + DMA_BIAS - 1024 i, base - DMA_BIAS).
    __device__ __forceinline__ void hm_loads(uint32_t m0, const void* base, const uint32_t (&v)[2])
    {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024"
                     :
                     : "s"(hd_scalar(m0)), "v"(v[0]), "v"(v[1]), "s"(hd_scalar(base))
                     : "memory");
    }
    __device__ __forceinline__ void hm_loads(uint32_t m0, const void* base, const uint32_t (&v)[4])
    {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %5 offset:1024\n\t"
                     "global_load_lds_dwordx4 %3, %5 offset:2048\n\tglobal_load_lds_dwordx4 %4, %5 offset:3072"
                     :
                     : "s"(hd_scalar(m0)), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(hd_scalar(base))
                     : "memory");
    }
    // 16 bytes per lane, each from an address of its own, to m0 + 16 * lane
    __device__ __forceinline__ void hm_load_at(uint32_t m0, const void* lane_address)
    {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(hd_scalar(m0)), "v"(lane_address) : "memory");
    }
    // One operand: its share of the loads, and its MFMA operand fetches (NB blocks of 16 rows per wave tile).
    template <bool KF, int BR, int NB>
    struct HmOperand
    {
        static constexpr int NL = BR / 32;
        uint32_t             voff[NL]; // byte offsets of this lane's loads from the tile's k origin (biased, see hm_loads)
        int                  frag[KF ? 2 : NB]; // element offsets of the MFMA operand fetches in a stage
        const char*          base;
        uint32_t             kb; // bytes between consecutive k

        __device__ inline void init(const void* ptr, const int32_t* rtab, int rstride, int r0, int rows, int kstride, int wave, int lane)
        {
            base = (const char*)ptr;
            kb   = 2u * (uint32_t)kstride;
#pragma unroll
            for(int i = 0; i < NL; i++)
            {
                const HdSlot s = hm_slot<KF, BR>((wave * NL + i) * 64 + lane);
                voff[i]        = 2u * row_offset(rtab, rstride, r0 + s.row, rows) + (uint32_t)s.k * kb + (uint32_t)(DMA_BIAS - (i % 4) * 1024);
            }
        }
        // (one row mode: computed, which spares the prologue a round trip to the table; rows beyond the last read
        // row 0, as the table has them)
        __device__ static inline uint32_t row_offset(const int32_t* rtab, int rstride, int r, int rows)
        {
            return rstride ? (r < rows ? (uint32_t)r * (uint32_t)rstride : 0u) : (uint32_t)rtab[r];
        }
        // the loads of the tile from k = ko on into the operand's stage at LDS address dst
        __device__ inline void request(uint32_t dst, int ko, int wave) const
        {
            hm_loads(dst + (uint32_t)wave * (NL * 1024u), base - DMA_BIAS + (uint64_t)((uint32_t)ko * kb), voff);
        }
        // ... of the tile of which only the first tail_k k lie inside K (chunks: see hm_tail_k)
        __device__ inline void request_tail(uint32_t dst, int ko, int tail_k, bool chunks, int wave, int lane) const
        {
            const char* origin = base + (uint64_t)((uint32_t)ko * kb);
#pragma unroll
            for(int i = 0; i < NL; i++)
            {
                const HdSlot s = hm_slot<KF, BR>((wave * NL + i) * 64 + lane);
                const int    k = hm_tail_k(s.k, tail_k, chunks);
                const char*  p = origin + (voff[i] - (uint32_t)(DMA_BIAS - (i % 4) * 1024)) - (int64_t)(s.k - k) * (int64_t)kb;
                hm_load_at(dst + (uint32_t)(wave * NL + i) * 1024u, k != HM_ZERO ? (const void*)p : (const void*)hm_zero16);
            }
        }
        // operand fetch of the 16-row block b from row `wrow` of the tile on, k-step ks (32 k): as HkFrag (contract_hk.hpp)
        __device__ inline void init_frag(int wrow, int lane)
        {
            if constexpr(KF)
            {
                const int row = wrow + (lane & 15);
#pragma unroll
                for(int ks = 0; ks < 2; ks++)
                    frag[ks] = row * HK_BK + (hk_chunk_pos(row, 4 * ks + (lane >> 4)) << 3);
            }
            else
            {
                const int k = 8 * (lane >> 4) + ((lane & 15) >> 2);
#pragma unroll
                for(int b = 0; b < NB; b++)
                    frag[b] = k * BR + hd_row_pos(wrow + 16 * b + 4 * (lane & 3), k);
            }
        }
        __device__ inline u32x4_t fetch(const uint16_t* stage, int b, int ks) const
        {
            if constexpr(KF)
                return *(const u32x4_t*)(stage + frag[ks] + b * 16 * HK_BK);
            else
            {
                typedef short4_t __attribute__((address_space(3))) * lds_s4_ptr;
                const uint16_t* p  = stage + frag[b] + ks * 32 * BR;
                const short4_t  lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_ptr)(p));
                const short4_t  hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_ptr)(p + 4 * BR));
                const u32x2_t   l2 = __builtin_bit_cast(u32x2_t, lo);
                const u32x2_t   h2 = __builtin_bit_cast(u32x2_t, hi);
                return u32x4_t{l2[0], l2[1], h2[0], h2[1]};
            }
        }
    };

    template <typename Tr, bool XKF, bool YKF, int BP, int BQ, int NS>
    __global__ void __launch_bounds__(256, 2) contract_hm_kernel(const KArgs a)
    {
        typedef HmGeom<BP, BQ, NS> G;
        constexpr int WP = G::WP, WQ = G::WQ, TP = G::TP, TQ = G::TQ, NBP = 2 * TP, NBQ = 2 * TQ, LPT = G::LPT;

        extern __shared__ __attribute__((aligned(16))) uint16_t lds[];

        const int tid  = threadIdx.x;
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wp   = wave / WQ;
        const int wq   = wave % WQ;

        int tp, tq, slice;
        tile_coords(a, tp, tq, slice);
        const int p_own = tp * BP, q_own = tq * BQ;
        const int p0    = (a.shift_p && p_own + BP > a.P) ? a.P - BP : p_own;
        const int q0    = (a.shift_q && q_own + BQ > a.Q) ? a.Q - BQ : q_own;

        const HmSlice sl = hm_slice(a.K, slice * a.ktiles_per_split, a.ktiles_per_split);

        typedef uint16_t __attribute__((address_space(3))) * lds_u16_ptr;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_u16_ptr)lds;

        HmOperand<XKF, BP, NBP> x;
        HmOperand<YKF, BQ, NBQ> y;
        x.init(a.X, a.xp, a.xp_stride, p0, a.P, a.xk_stride, wave, lane);
        y.init(a.Y, a.yq, a.yq_stride, q0, a.Q, a.yk_stride, wave, lane);
        x.init_frag(wp * TP * 32, lane);
        y.init_frag(wq * TQ * 32, lane);

        auto request = [&](int u, int stage) __attribute__((always_inline)) {
            const uint32_t dst = lds0 + (uint32_t)stage * (G::STAGE * 2u);
            const int      ko  = hm_origin(sl, u);
            x.request(dst, ko, wave);
            y.request(dst + G::OPX * 2u, ko, wave);
        };

        f32x4_t acc[NBP][NBQ];
#pragma unroll
        for(int i = 0; i < NBP; i++)
#pragma unroll
            for(int j = 0; j < NBQ; j++)
                acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

        // this wave's MFMA operands of one K tile: tile t + 1's are read from LDS while tile t is multiplied
        struct Frags
        {
            u32x4_t x[2][NBP], y[2][NBQ];
        };
        Frags f0, f1;
        auto  read_tile = [&](int stage, Frags& f) __attribute__((always_inline)) {
            const uint16_t* sx = lds + stage * G::STAGE;
            const uint16_t* sy = sx + G::OPX;
#pragma unroll
            for(int ks = 0; ks < 2; ks++)
            {
#pragma unroll
                for(int i = 0; i < NBP; i++)
                    f.x[ks][i] = x.fetch(sx, i, ks);
#pragma unroll
                for(int j = 0; j < NBQ; j++)
                    f.y[ks][j] = y.fetch(sy, j, ks);
            }
        };
        auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
            for(int ks = 0; ks < 2; ks++)
#pragma unroll
                for(int i = 0; i < NBP; i++)
#pragma unroll
                    for(int j = 0; j < NBQ; j++)
                        acc[i][j] = hk_mfma16(Tr{}, f.x[ks][i], f.y[ks][j], acc[i][j]);
        };
        // tile t, in `cur`; BEHIND: tiles on their way behind tile t + 1, which must have landed
        int  t = 0, stage = 0;
        auto step = [&](auto behind_c, bool more, const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(decltype(behind_c)::value * LPT));
            lds_barrier();
            // every wave has tile t in registers: its stage is free
            const int next = stage + 1 == NS ? 0 : stage + 1;
            read_tile(next, nxt);
            __builtin_amdgcn_sched_barrier(0);
            if(more)
                request(t + NS, stage);
            multiply(cur);
            __builtin_amdgcn_sched_barrier(0);
            stage = next;
            t++;
        };
        // the last tiles, behind which fewer than NS - 1 are on their way
        auto last_steps = [&](const Frags& cur, Frags& nxt) __attribute__((always_inline)) {
            const int  behind = sl.nt - 2 - t;
            const bool more   = t + NS < sl.nt;
            if(behind >= NS - 2)
                step(std::integral_constant<int, NS - 2>{}, more, cur, nxt);
            else if(NS > 3 && behind == 1)
                step(std::integral_constant<int, 1>{}, false, cur, nxt);
            else if(behind == 0)
                step(std::integral_constant<int, 0>{}, false, cur, nxt);
            else
            {
                multiply(cur);
                t++;
            }
        };

        // the first NS tiles; the first of them has landed when only the others are on their way
        if(sl.tail_k)
        {
            const int ko = hm_origin(sl, 0);
            x.request_tail(lds0, ko, sl.tail_k, XKF || YKF, wave, lane);
            y.request_tail(lds0 + G::OPX * 2u, ko, sl.tail_k, XKF || YKF, wave, lane);
        }
        else
            request(0, 0);
#pragma unroll
        for(int u = 1; u < NS; u++)
            if(u < sl.nt)
                request(u, u);
        if(sl.nt >= NS)
            __builtin_amdgcn_s_waitcnt(waitcnt_vm((NS - 1) * LPT));
        else
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        lds_barrier();
        read_tile(0, f0);
        if((XKF || YKF) && sl.tail_k % 8 != 0)
        {
            // the eight k that K ends in are the last eight of K: those that the chunk in front of them holds as well
            // count once
            const int dup = 8 - sl.tail_k % 8; // (even)
#pragma unroll
            for(int ks = 0; ks < 2; ks++)
            {
                const bool mine = 4 * ks + (lane >> 4) == sl.tail_k / 8;
                u32x4_t    keep;
#pragma unroll
                for(int e = 0; e < 4; e++)
                    keep[e] = mine && 2 * e < dup ? 0u : 0xFFFFFFFFu;
#pragma unroll
                for(int i = 0; i < NBP; i++)
                    f0.x[ks][i] &= keep;
#pragma unroll
                for(int j = 0; j < NBQ; j++)
                    f0.y[ks][j] &= keep;
            }
        }
        while(t + 1 + NS < sl.nt)
        {
            step(std::integral_constant<int, NS - 2>{}, true, f0, f1);
            step(std::integral_constant<int, NS - 2>{}, true, f1, f0);
        }
        while(t < sl.nt)
        {
            last_steps(f0, f1);
            if(t < sl.nt)
                last_steps(f1, f0);
        }
        // (the epilogue stages through this LDS)
        lds_barrier();
        epilogue_h16<Tr, WP, WQ, TP, TQ, G::LDS_BYTES>(a, acc, lds, p0, q0, p_own, q_own, slice);
    }

    template <typename Tr, bool XKF, bool YKF, int BP, int BQ, int NS>
    int launch_hm(const KArgs& a, hipStream_t stream)
    {
        typedef HmGeom<BP, BQ, NS> G;
        if(((XKF || YKF) && a.K % 2 != 0) || (a.shift_p && a.P < BP) || (a.shift_q && a.Q < BQ))
            return (int)hipErrorInvalidValue;
        auto                    kern = contract_hm_kernel<Tr, XKF, YKF, BP, BQ, NS>;
        static const hipError_t attr = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS_BYTES);
        if(attr != hipSuccess)
            return (int)attr;
        dim3 grid(a.tiles_p * a.tiles_q, 1, a.split_k);
        hipLaunchKernelGGL(kern, grid, dim3(256), G::LDS_BYTES, stream, a);
        return (int)hipGetLastError();
    }
}

// Registry lines: operands gathered in 16-byte vectors that start at multiples of 4 bytes, one k stride each; K even
// if an operand is contiguous along it.
#define HIPTK_HM_ENTRY(TR, ID, BP, BQ, XKF, YKF, NS)                                                        \
    {                                                                                                       \
        TR::CLS, ID, XKF, YKF, 8, 8, true, BP, BQ, 64, 256, hiptk::HmGeom<BP, BQ, NS>::LDS_BYTES,            \
            #TR "_" #BP "x" #BQ "x64_x" #XKF "8_y" #YKF "8_kafftrue_direct_ring" #NS,                       \
            &hiptk::launch_hm<hiptk::TR, XKF, YKF, BP, BQ, NS>, (XKF || YKF) ? 2 : 1, 32, 4                    \
    }
#define HIPTK_HM_TILE(TR, ID, BP, BQ, NS)                                                                   \
    HIPTK_HM_ENTRY(TR, ID, BP, BQ, true, true, NS), HIPTK_HM_ENTRY(TR, ID, BP, BQ, true, false, NS),         \
        HIPTK_HM_ENTRY(TR, ID, BP, BQ, false, true, NS), HIPTK_HM_ENTRY(TR, ID, BP, BQ, false, false, NS)
