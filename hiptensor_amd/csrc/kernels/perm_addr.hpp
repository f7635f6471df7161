// Address arithmetic of the permutation kernels that move 16-byte vectors at any element (the linear kernel and the
// grouped tiles, permute.hip), in functions that also compile for the host: such vectors start anywhere and the last of
// a run is moved back to end with it, so every load and store of every thread is walked on the CPU
// (tests/cpp/perm_bounds.cpp).
#pragma once
#include <stdint.h>

#include <algorithm>

#include "hiptk_kernels.h"

#if defined(__HIPCC__)
#define HIPTK_PERM_FN __host__ __device__ inline
#else
#define HIPTK_PERM_FN inline
#endif

namespace hiptk
{
    constexpr int PERM_THREADS = 256;
    constexpr int PERM_BATCH   = HIPTK_PERM_MAX_RANK - 2;

    HIPTK_PERM_FN uint32_t mul_hi(uint32_t x, uint32_t y)
    {
        return (uint32_t)(((uint64_t)x * y) >> 32);
    }

    // floor(2^32 / d) + 1, d >= 2: mul_hi(v, magic_of(d)) == v / d while v * d < 2^32
    inline uint32_t magic_of(uint32_t d)
    {
        return (uint32_t)((uint64_t(1) << 32) / d) + 1u;
    }

    // 2^32 / d rounded up, d >= 2: mul_hi(v, recip(d)) == v / d while v * d < 2^32
    HIPTK_PERM_FN uint32_t recip(uint32_t d)
    {
        return 0xFFFFFFFFu / d + 1u;
    }

    // x / e and x % e by the reciprocal m = floor(2^32 / e) + 1, exact for every 32-bit x (the high word is the
    // quotient or one more)
    HIPTK_PERM_FN uint32_t div_by(uint32_t x, uint32_t e, uint32_t m, uint32_t& rem)
    {
        uint32_t q = mul_hi(x, m), r = x - q * e;
        if((int32_t)r < 0)
        {
            q -= 1;
            r += e;
        }
        rem = r;
        return q;
    }

    // ---------------------------------------------------------------- linear kernel (HIPTK_PERM_RUNS)

    struct RunsShape
    {
        uint32_t n; // elements
        uint32_t e0, m0; // extent of the shared fastest mode and its reciprocal
        int32_t  nb; // the other modes, in B's order
        uint32_t ext[HIPTK_PERM_MAX_RANK - 1], astr[HIPTK_PERM_MAX_RANK - 1], magic[HIPTK_PERM_MAX_RANK - 1];
    };

    inline RunsShape runs_shape(const hiptk_permute_t& p, int64_t n)
    {
        RunsShape a = {};
        a.n         = (uint32_t)n;
        a.e0        = (uint32_t)p.extent[0];
        a.m0        = magic_of(a.e0);
        int order[HIPTK_PERM_MAX_RANK];
        for(int d = 0; d < p.rank; ++d)
            order[d] = d;
        std::sort(order + 1, order + p.rank, [&p](int x, int y) {
            return p.b_stride[x] != p.b_stride[y] ? p.b_stride[x] < p.b_stride[y] : x < y;
        });
        for(int k = 1; k < p.rank; ++k)
        {
            const int d = order[k];
            if(p.extent[d] == 1)
                continue;
            a.ext[a.nb]   = (uint32_t)p.extent[d];
            a.astr[a.nb]  = (uint32_t)p.a_stride[d];
            a.magic[a.nb] = magic_of((uint32_t)p.extent[d]);
            ++a.nb;
        }
        return a;
    }

    // Vectors per thread.  Four keep more loads in flight, but a tensor of a few MB then makes too few workgroups for
    // 256 compute units and the kernel lasts as long as one thread (2^17 f32: 32 workgroups): f32
    // 16.20.4.8.8.4 -> (0,1,4,3,5,2) 5.7 us, 3.9 in tiles; one per thread takes 0.58-0.75 of four's time up to 2^20
    // f32 (0.60-0.72 up to 2^21 f16), 0.87-0.91 just below the line here and 0.94-1.02 beyond it, with cases of up
    // to 1.24.  From four workgroups of four a compute unit on, four.
    inline int runs_per_thread(int64_t n, int v)
    {
        return n >= (int64_t(1) << 20) * v ? 4 : 1;
    }

    // Where the V elements of B from idx on lie in A: those of this run from src on, those of the next from next on, so
    // that V from src and V from next - left hold them.  Neither reaches beyond the ends of A, whose first and last
    // runs are B's as well: a run that ends with A has no next one, and a next one does not start at 0.
    struct RunsVector
    {
        uint32_t src, next, left; // left: elements of this run from src on
    };

    HIPTK_PERM_FN RunsVector runs_vector(const RunsShape& a, uint32_t idx)
    {
        uint32_t pos, off = 0, noff = 0;
        uint32_t rem   = div_by(idx, a.e0, a.m0, pos);
        bool     carry = true; // the next run's coordinates: one more, from the fastest mode up
        for(int d = 0; d < a.nb; ++d)
        {
            uint32_t c;
            rem = div_by(rem, a.ext[d], a.magic[d], c);
            const uint32_t c1 = !carry ? c : c + 1 == a.ext[d] ? 0u : c + 1;
            off += c * a.astr[d];
            noff += c1 * a.astr[d];
            carry = carry && c1 == 0;
        }
        RunsVector r;
        r.src  = off + pos;
        r.next = noff;
        r.left = a.e0 - pos;
        return r;
    }

    // ---------------------------------------------------------------- plain tiles (HIPTK_PERM_TILED)

    // The part of the work workgroup `b` of `n` takes: with `bands`, workgroups of one die (ids that are congruent mod 8)
    // take neighbouring parts.
    HIPTK_PERM_FN uint32_t tile_work(uint32_t b, uint32_t n, bool bands)
    {
        if(!bands)
            return b;
        const uint32_t die = b & 7, rem = n & 7;
        return die * (n >> 3) + (die < rem ? die : rem) + (b >> 3);
    }

    // First element along both tile modes of the work-th tile, and its offsets in A and B.
    // Workgroups that run at the same time should spread over both tile modes: tiles that are neighbours along i touch
    // neighbouring addresses of A, neighbours along j neighbouring addresses of B.  The tile plane is cut into bands of
    // `group` tiles along j; inside a band the walk is j-first.
    template <typename Args>
    HIPTK_PERM_FN void tile_origin(const Args& a, uint32_t work, uint32_t TI, uint32_t TJ, uint32_t& i0, uint32_t& j0, uint32_t& aoff, uint32_t& boff)
    {
        const uint32_t plane = a.nt_i * a.nt_j;
        uint32_t       blk   = work / plane;
        const uint32_t lin   = work - blk * plane;
        uint32_t       ti, tj;
        if(a.group == 0)
        {
            // diagonal walk: consecutive workgroups differ in both tile coordinates, so that
            // with power-of-two strides neither side keeps hitting the same memory channels
            ti                = lin % a.nt_i;
            const uint32_t rj = lin / a.nt_i;
            tj                = (rj + ti) % a.nt_j;
        }
        else
        {
            const uint32_t band = lin / (a.group * a.nt_i);
            const uint32_t rem  = lin - band * (a.group * a.nt_i);
            const uint32_t left = a.nt_j - band * a.group;
            const uint32_t rows = left < a.group ? left : a.group;
            ti                  = rem / rows;
            tj                  = band * a.group + (rem - ti * rows);
        }
        aoff = 0;
        boff = 0;
        for(int d = 0; d < a.nb; ++d)
        {
            const uint32_t c = blk % a.bext[d];
            blk /= a.bext[d];
            aoff += c * a.ba[d];
            boff += c * a.bb[d];
        }
        i0 = ti * TI;
        j0 = tj * TJ;
        aoff += i0 + j0 * a.a_j;
        boff += i0 * a.b_i + j0 * a.b_j;
    }

    // Vector v of a tile's `lines` rows (columns) of n elements, W elements of `per_line` vectors a line: the line and the
    // first element along it.
    struct TileVector
    {
        bool     ok; // inside the tile
        uint32_t line, at;
    };

    // (LOOSE: the last vector of a line is moved back to end with it; n is W at least)
    template <int W, bool LOOSE>
    HIPTK_PERM_FN TileVector tile_vector(uint32_t v, uint32_t per_line, uint32_t n, uint32_t lines)
    {
        TileVector r;
        r.line = v / per_line;
        r.at   = (v - r.line * per_line) * W;
        r.ok   = r.at < n && r.line < lines;
        if(LOOSE)
            r.at = r.at + W > n ? n - W : r.at;
        return r;
    }

    // ---------------------------------------------------------------- grouped tiles (HIPTK_PERM_GROUPED)

    struct GroupShape
    {
        uint32_t e_i0, e_i1, e_j0, e_j1; // extents of the row modes (0, i2) and the column modes (j, j2); 1 if absent
        uint32_t w_i, w_j; // elements of mode 0 / mode j per tile (== the extent when c > 1)
        uint32_t c_i, c_j; // indices of i2 / j2 per tile
        uint32_t a_j0, a_j1, b_i0, b_i1; // A strides of the column modes, B strides of the row modes
        uint32_t nt_i0, nt_j0, nt_i, nt_j; // tiles along mode 0, mode j, i2 and j2
        uint32_t pitch; // LDS row pitch in elements: an odd number of 32-bit words
        uint32_t m_rv, m_wj, m_cv, m_wi; // floor(2^32 / d) + 1 for d = vectors per row, w_j, vectors per column, w_i
        int32_t  nb;
        uint32_t bext[PERM_BATCH], ba[PERM_BATCH], bb[PERM_BATCH];
    };

    // (of a problem whose modes, widths and chunks have been checked)
    inline GroupShape group_shape(const hiptk_permute_t& p, int64_t& grid)
    {
        const int  mj = p.mode_j, mi2 = p.mode_i2, mj2 = p.mode_j2;
        GroupShape a = {};
        a.e_i0       = (uint32_t)p.extent[0];
        a.e_i1       = mi2 == -1 ? 1u : (uint32_t)p.extent[mi2];
        a.e_j0       = (uint32_t)p.extent[mj];
        a.e_j1       = mj2 == -1 ? 1u : (uint32_t)p.extent[mj2];
        a.w_i        = (uint32_t)p.width_i;
        a.w_j        = (uint32_t)p.width_j;
        a.c_i        = (uint32_t)p.chunk_i;
        a.c_j        = (uint32_t)p.chunk_j;
        a.a_j0       = (uint32_t)p.a_stride[mj];
        a.a_j1       = mj2 == -1 ? 0u : (uint32_t)p.a_stride[mj2];
        a.b_i0       = (uint32_t)p.b_stride[0];
        a.b_i1       = mi2 == -1 ? 0u : (uint32_t)p.b_stride[mi2];
        a.nt_i0      = (a.e_i0 + a.w_i - 1) / a.w_i;
        a.nt_j0      = (a.e_j0 + a.w_j - 1) / a.w_j;
        a.nt_i       = (a.e_i1 + a.c_i - 1) / a.c_i;
        a.nt_j       = (a.e_j1 + a.c_j - 1) / a.c_j;
        const uint32_t TI = a.w_i * a.c_i, TJ = a.w_j * a.c_j;
        const uint32_t wordElems  = 4u / (uint32_t)p.elem_bytes; // elements per 32-bit word
        uint32_t       pitchWords = (TI + wordElems - 1) / wordElems;
        pitchWords |= 1u; // odd: consecutive rows start in different banks
        a.pitch           = pitchWords * wordElems;
        const uint32_t vr = (uint32_t)p.vec_r, vw = (uint32_t)p.vec_w;
        a.m_rv            = magic_of(p.loose ? (TI + vr - 1) / vr : TI / vr);
        a.m_wj            = magic_of(a.w_j);
        a.m_cv            = magic_of(p.loose ? (TJ + vw - 1) / vw : TJ / vw);
        a.m_wi            = magic_of(a.w_i);
        grid              = (int64_t)a.nt_i0 * a.nt_j0 * a.nt_i * a.nt_j;
        for(int d = 1; d < p.rank; ++d)
        {
            if(d == mj || d == mi2 || d == mj2)
                continue;
            a.bext[a.nb] = (uint32_t)p.extent[d];
            a.ba[a.nb]   = (uint32_t)p.a_stride[d];
            a.bb[a.nb]   = (uint32_t)p.b_stride[d];
            ++a.nb;
            grid *= p.extent[d];
        }
        return a;
    }

    // A workgroup's tile: where it starts, and the rows and columns of it that lie inside the extents.
    struct GroupTile
    {
        uint32_t aoff, boff, nx, ny;
    };

    HIPTK_PERM_FN GroupTile group_tile(const GroupShape& a, uint32_t blk)
    {
        const uint32_t ti0 = blk % a.nt_i0;
        blk /= a.nt_i0;
        const uint32_t tj0 = blk % a.nt_j0;
        blk /= a.nt_j0;
        const uint32_t ti = blk % a.nt_i;
        blk /= a.nt_i;
        const uint32_t tj = blk % a.nt_j;
        blk /= a.nt_j;
        GroupTile t;
        t.aoff = t.boff = 0;
        for(int d = 0; d < a.nb; ++d)
        {
            const uint32_t c = blk % a.bext[d];
            blk /= a.bext[d];
            t.aoff += c * a.ba[d];
            t.boff += c * a.bb[d];
        }
        const uint32_t i0s = ti0 * a.w_i, j0s = tj0 * a.w_j;
        const uint32_t wi = (a.e_i0 - i0s) < a.w_i ? (a.e_i0 - i0s) : a.w_i;
        const uint32_t wj = (a.e_j0 - j0s) < a.w_j ? (a.e_j0 - j0s) : a.w_j;
        const uint32_t i1s = ti * a.c_i, j1s = tj * a.c_j;
        const uint32_t ci = (a.e_i1 - i1s) < a.c_i ? (a.e_i1 - i1s) : a.c_i;
        const uint32_t cj = (a.e_j1 - j1s) < a.c_j ? (a.e_j1 - j1s) : a.c_j;
        // (c > 1 only with the whole first mode: w == e)
        t.nx = a.w_i * (ci - 1) + wi;
        t.ny = a.w_j * (cj - 1) + wj;
        t.aoff += i0s + i1s * a.e_i0 + j0s * a.a_j0 + j1s * a.a_j1;
        t.boff += i0s * a.b_i0 + i1s * a.b_i1 + j0s + j1s * a.e_j0;
        return t;
    }

    // Vector v of a tile's rows (columns), W elements of `per_line` vectors a line: the line, the first element along
    // it, and the line's offset in A (B) from the tile's start.
    struct GroupVector
    {
        bool     ok; // inside the tile
        uint32_t line, at, off;
    };

    template <int W, bool LOOSE>
    HIPTK_PERM_FN GroupVector group_read(const GroupShape& a, const GroupTile& t, uint32_t v, uint32_t per_line, uint32_t magic)
    {
        GroupVector r;
        r.line            = mul_hi(v, magic);
        r.at              = (v - r.line * per_line) * W;
        const uint32_t y1 = mul_hi(r.line, a.m_wj), y0 = r.line - y1 * a.w_j;
        r.ok              = v < per_line * t.ny && r.at < t.nx;
        if(LOOSE)
            r.at = r.at + W > t.nx ? t.nx - W : r.at;
        r.off = y0 * a.a_j0 + y1 * a.a_j1;
        return r;
    }

    template <int W, bool LOOSE>
    HIPTK_PERM_FN GroupVector group_write(const GroupShape& a, const GroupTile& t, uint32_t v, uint32_t per_line, uint32_t magic)
    {
        GroupVector r;
        r.line = mul_hi(v, magic);
        r.at   = (v - r.line * per_line) * W;
        r.ok   = r.at < t.ny;
        if(LOOSE)
            r.at = r.at + W > t.ny ? t.ny - W : r.at;
        const uint32_t x1 = mul_hi(r.line, a.m_wi), x0 = r.line - x1 * a.w_i;
        r.off             = x0 * a.b_i0 + x1 * a.b_i1;
        return r;
    }

    // vectors per nominal row / column
    HIPTK_PERM_FN uint32_t group_per_line(uint32_t elems, uint32_t v, bool loose)
    {
        return (elems + (loose ? v - 1 : 0)) / v;
    }

    // single elements of a line shorter than a vector: their number, 2 at least as the reciprocal wants it
    HIPTK_PERM_FN uint32_t group_singles(uint32_t n)
    {
        return n < 2 ? 2 : n;
    }
}
