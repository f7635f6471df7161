#include "permute_plan.hpp"

#include <algorithm>
#include <cstring>

namespace hipta
{
    namespace
    {
        struct Tile
        {
            int ti, tj;
        };
        // the kernel layer's tile shapes (elements): square, long along i, long along j
        constexpr Tile TILES4[4] = {{64, 64}, {256, 16}, {16, 256}, {128, 128}};
        constexpr Tile TILES2[4] = {{128, 128}, {512, 32}, {32, 512}, {256, 128}};

        bool alignedTo(const void* p, int64_t bytes)
        {
            return (reinterpret_cast<uintptr_t>(p) % (uintptr_t)bytes) == 0;
        }

        // Largest vector (elements) not above cap that divides `extent` and every stride in
        // `others`, and that the address is aligned for.
        int pickVec(int elem_bytes, int cap, int64_t extent, const std::vector<int64_t>& others, const void* p, bool copy)
        {
            const int cands4[] = {4, 2, 1}, cands2[] = {8, 2, 1}, candsCopy2[] = {8, 4, 2, 1};
            const int* c;
            int        n;
            if(elem_bytes == 4)
                c = cands4, n = 3;
            else if(copy)
                c = candsCopy2, n = 4;
            else
                c = cands2, n = 3;
            for(int k = 0; k < n; ++k)
            {
                const int v = c[k];
                if(v > cap || extent % v != 0 || !alignedTo(p, (int64_t)v * elem_bytes))
                    continue;
                bool ok = true;
                for(int64_t s : others)
                    ok = ok && (s % v == 0);
                if(ok)
                    return v;
            }
            return 1;
        }

        // Share of a tile grid's lanes that fall inside the extents.
        double coverage(int64_t e, int t)
        {
            const int64_t tiles = (e + t - 1) / t;
            return (double)e / (double)(tiles * t);
        }

        int pickTile(int elem_bytes, int64_t e_i, int64_t e_j, const int order[3])
        {
            const Tile* ts   = elem_bytes == 4 ? TILES4 : TILES2;
            int         best = order[0];
            double      bc   = -1.0;
            for(int k = 0; k < 3; ++k)
            {
                const int    t = order[k];
                const double c = coverage(e_i, ts[t].ti) * coverage(e_j, ts[t].tj);
                if(c > bc + 1e-9)
                    bc = c, best = t;
            }
            return best;
        }
    }

    static PermuteStatus pick_kernel(const PermuteIn& in, const PermuteTuning& tune, hiptk_permute_t& out)
    {
        std::memset(&out, 0, sizeof(out));
        const size_t rank = in.lenA.size();
        if(in.lenB.size() != rank || in.modeA.size() != rank || in.modeB.size() != rank)
            return PermuteStatus::BAD_RANK;

        // position of each B mode in A; every label once on both sides, lengths agree
        std::vector<int> posInA(rank, -1);
        std::vector<bool> used(rank, false);
        for(size_t k = 0; k < rank; ++k)
        {
            for(size_t i = 0; i < rank; ++i)
                if(in.modeA[i] == in.modeB[k] && !used[i])
                {
                    posInA[k] = (int)i;
                    break;
                }
            if(posInA[k] < 0 || in.lenB[k] != in.lenA[posInA[k]])
                return PermuteStatus::BAD_MODES;
            used[posInA[k]] = true;
        }
        int64_t count = 1;
        for(size_t i = 0; i < rank; ++i)
        {
            if(in.lenA[i] < 0)
                return PermuteStatus::BAD_MODES;
            if(in.lenA[i] == 0)
                return PermuteStatus::EMPTY;
            count *= in.lenA[i];
            if(count >= (int64_t(1) << 31))
                return PermuteStatus::TOO_LARGE;
        }

        // packed strides, first listed mode fastest; B's stride carried to A's order
        std::vector<int64_t> bInA(rank, 0);
        {
            int64_t s = 1;
            for(size_t k = 0; k < rank; ++k)
            {
                bInA[posInA[k]] = s;
                s *= in.lenB[k];
            }
        }
        // drop extent-1 modes, fuse neighbours of A that are neighbours in B in the same order
        std::vector<int64_t> ext, as, bs;
        {
            int64_t s = 1;
            for(size_t i = 0; i < rank; ++i)
            {
                const int64_t e = in.lenA[i];
                if(e != 1)
                {
                    if(!ext.empty() && bInA[i] == bs.back() * ext.back())
                        ext.back() *= e;
                    else
                    {
                        ext.push_back(e);
                        as.push_back(s);
                        bs.push_back(bInA[i]);
                    }
                }
                s *= e;
            }
            if(ext.empty())
            {
                ext.push_back(1);
                as.push_back(1);
                bs.push_back(1);
            }
        }
        const int r    = (int)ext.size();
        if(r > HIPTK_PERM_MAX_RANK)
            return PermuteStatus::BAD_RANK; // more modes left after fusion than the kernels index
        out.elem_bytes = in.elem_bytes;
        out.rank       = r;
        for(int d = 0; d < r; ++d)
        {
            out.extent[d]   = (int32_t)ext[d];
            out.a_stride[d] = (int32_t)as[d];
            out.b_stride[d] = (int32_t)bs[d];
        }
        out.vec_r = out.vec_w = 1;
        out.group             = tune.group >= 0 ? tune.group : 1;
        const int cap         = std::max(1, tune.max_vec);

        if(r == 1)
        {
            out.kernel = HIPTK_PERM_COPY;
            const int v = std::min(pickVec(in.elem_bytes, cap, ext[0], {}, in.A, true),
                                   pickVec(in.elem_bytes, cap, ext[0], {}, in.B, true));
            out.vec_r = out.vec_w = v;
            return PermuteStatus::OK;
        }

        int jB = 0; // B's fastest mode
        for(int d = 0; d < r; ++d)
            if(bs[d] == 1)
                jB = d;

        // layout-admissible kernels: TILED needs differing fastest modes, ROWS a shared one,
        // STRIP a tile mode of at most 64 elements whose partner follows it directly in memory
        const bool shared = jB == 0;
        const bool stripJ = !shared && ext[jB] <= 64 && ext[jB] <= ext[0] && bs[0] == ext[jB]; // short j, B holds i right after it
        const bool stripI = !shared && ext[0] <= 64 && jB == 1 && !stripJ; // short i, A holds j right after it
        // Many short modes: no single mode gives a long run.  A tile row then spans A's two
        // fastest modes and a tile column B's two fastest modes, where those are free.
        // Fills `out` and returns true when that kernel applies (force: even where the plain
        // tiles would cover the extents well).
        auto tryGrouped = [&](bool force, bool anySize) -> bool {
            if(shared)
                return false;
            const int64_t target = 128; // elements per tile row / column aimed at
            // a side whose fastest mode is short takes a chunk of the next mode along; a long one
            // is tiled by itself
            int mi2 = (ext[0] <= target && r > 1 && jB != 1) ? 1 : -1;
            int mj2 = -1;
            if(ext[jB] <= target)
                for(int d = 1; d < r; ++d)
                    if(bs[d] == ext[jB])
                        mj2 = d;
            if(mi2 != -1 && mi2 == mj2) // both sides want mode 1: the side with the shorter run gets it
                (ext[jB] < ext[0] ? mi2 : mj2) = -1;
            const int    order[] = {0, 1, 2};
            const int    st      = pickTile(in.elem_bytes, ext[0], ext[jB], order);
            const Tile*  ts      = in.elem_bytes == 4 ? TILES4 : TILES2;
            const double cov     = coverage(ext[0], ts[st].ti) * coverage(ext[jB], ts[st].tj);
            if(cov >= 0.7 && !force)
                return false;
            std::vector<int64_t> aOth(as.begin() + 1, as.end()), bOth;
            for(int d = 0; d < r; ++d)
                if(d != jB)
                    bOth.push_back(bs[d]);
            int vr = pickVec(in.elem_bytes, cap, ext[0], aOth, in.A, false);
            int vw = pickVec(in.elem_bytes, cap, ext[jB], bOth, in.B, false);
            int64_t wi = std::min<int64_t>(ext[0], target), wj = std::min<int64_t>(ext[jB], target);
            int64_t ci = mi2 == -1 ? 1 : std::max<int64_t>(1, std::min<int64_t>(ext[mi2], target / ext[0]));
            int64_t cj = mj2 == -1 ? 1 : std::max<int64_t>(1, std::min<int64_t>(ext[mj2], target / ext[jB]));
            auto ldsBytes = [&]() { return (wj * cj) * (wi * ci + 2) * in.elem_bytes; };
            while(ldsBytes() > 56 * 1024)
            {
                // shrink the longer side: first its chunk, then (a tiled side) its width
                const bool iSide = wi * ci >= wj * cj;
                int64_t&   c     = iSide ? ci : cj;
                int64_t&   w     = iSide ? wi : wj;
                const int  v     = iSide ? vr : vw;
                if(c > 1)
                    c -= 1;
                else if(w > 2 * v && w > 16)
                    w = (w / 2 + v - 1) / v * v;
                else
                    return false;
            }
            // a small problem needs more workgroups than long runs: halve the larger side of the
            // tile until there are two workgroups per compute unit (256 of them) or the tile is small
            auto groups = [&]() {
                int64_t g = ((ext[0] + wi - 1) / wi) * ((ext[jB] + wj - 1) / wj);
                for(int d = 1; d < r; ++d)
                {
                    if(d == jB)
                        continue;
                    g *= d == mi2 ? (ext[d] + ci - 1) / ci : d == mj2 ? (ext[d] + cj - 1) / cj : ext[d];
                }
                return g;
            };
            while(groups() < 512 && wi * ci * wj * cj >= 2 * 2048)
            {
                const bool iSide = wi * ci >= wj * cj;
                int64_t&   c     = iSide ? ci : cj;
                int64_t&   w     = iSide ? wi : wj;
                const int  v     = iSide ? vr : vw;
                if(c > 1)
                    c = (c + 1) / 2;
                else if(w > 2 * v && w > 16)
                    w = (w / 2 + v - 1) / v * v;
                else
                    break;
            }
            while(vr > 1 && (wi * ci / vr < 2 || wi % vr != 0))
                vr = vr == 8 ? 2 : vr / 2;
            while(vw > 1 && (wj * cj / vw < 2 || wj % vw != 0))
                vw = vw == 8 ? 2 : vw / 2;
            if(wi < 2 || wj < 2 || wi * ci / vr < 2 || wj * cj / vw < 2)
                return false;
            if(wi * ci * wj * cj < 1536 && !anySize)
                return false; // tiles of a few hundred elements: one thread per element does better
                              // (192-element tiles: 459 against 1910 GB/s; 1890-element tiles: 1590 against 1190)
            out.kernel  = HIPTK_PERM_GROUPED;
            out.mode_i  = 0;
            out.mode_j  = jB;
            out.mode_i2 = mi2;
            out.mode_j2 = mj2;
            out.chunk_i = (int32_t)ci;
            out.chunk_j = (int32_t)cj;
            out.width_i = (int32_t)wi;
            out.width_j = (int32_t)wj;
            out.vec_r   = vr;
            out.vec_w   = vw;
            // Where the extents would leave narrow vectors: 16-byte ones at any element, if both sides of the tile are
            // 64 elements or more (f16 126 x 125 43.4 -> 29.4 us, 128 x 65 14.2 -> 8.4, f32 105 x 125 53.6 -> 43.0; but f16
            // 120 x 51 257 -> 278: the vector moved back at a short run's end weighs more).  Pairs of f16 are 4-byte
            // accesses already: they lose to it only while the tensor fits the L2 and the accesses are what counts (up
            // to 2^23 elements 0.70-0.98 of the pairs' time; beyond, 188 random shapes 0.68-1.57, half of them slower:
            // 138.16.70.18.82 -> (2,1,4,0,3) 388 us in pairs, 537 loose).  A side of single elements is worth it at any
            // size (0.51-1.0), next to pairs on the other side from columns of 120 elements on (0.55-0.99; shorter
            // ones 0.72-1.20).  f32 gains over the whole range (0.73-1.04).
            const int  full   = 16 / in.elem_bytes;
            const int  narrow = std::min(vr, vw), wide = std::max(vr, vw);
            const bool gains  = in.elem_bytes == 4 || count <= (1 << 23) || (narrow == 1 && (wide != 2 || wj * cj >= 120));
            if(cap >= full && narrow < full && wi * ci >= 64 && wj * cj >= 64 && gains)
            {
                out.loose = 1;
                out.vec_r = out.vec_w = full;
            }
            return true;
        };
        // A short shared fastest mode (interleaved channels): tiles of that mode times a chunk of
        // A's next mode times a chunk of B's next mode, so that both sides see long runs.
        auto tryShared = [&](bool force) -> bool {
            if(!shared || r < 3 || ext[0] > 128)
                return false;
            if(ext[0] * in.elem_bytes >= 64 && !force)
                return false; // from 64-byte runs on, plain rows do as well or better (measured)
            const int mi2 = 1;
            int       mj2 = -1;
            for(int d = 1; d < r; ++d)
                if(bs[d] == ext[0])
                    mj2 = d;
            if(mj2 == -1 || mj2 == mi2)
                return false;
            const int64_t target = 512 / in.elem_bytes; // elements per run aimed at
            int64_t       ci = std::max<int64_t>(1, std::min<int64_t>(ext[mi2], target / ext[0]));
            int64_t       cj = std::max<int64_t>(1, std::min<int64_t>(ext[mj2], target / ext[0]));
            auto ldsBytes = [&]() { return cj * (ext[0] * ci + 2) * in.elem_bytes; };
            while(ldsBytes() > 56 * 1024 && cj > 1)
                cj -= 1;
            if(ldsBytes() > 56 * 1024)
                return false;
            std::vector<int64_t> aOth(as.begin() + 1, as.end()), bOth(bs.begin() + 1, bs.end());
            int v = std::min(pickVec(in.elem_bytes, cap, ext[0], aOth, in.A, false), pickVec(in.elem_bytes, cap, ext[0], bOth, in.B, false));
            while(v > 1 && (ext[0] * ci / v < 2 || ext[0] * cj / v < 2))
                v = v == 8 ? 2 : v / 2;
            if(ext[0] * ci / v < 2 || ext[0] * cj / v < 2)
                return false;
            out.kernel  = HIPTK_PERM_SHARED;
            out.mode_i  = 0;
            out.mode_j  = 0;
            out.mode_i2 = mi2;
            out.mode_j2 = mj2;
            out.chunk_i = (int32_t)ci;
            out.chunk_j = (int32_t)cj;
            out.vec_r = out.vec_w = v;
            return true;
        };
        out.mode_i2 = out.mode_j2 = -1;
        out.chunk_i = out.chunk_j = 1;
        // Kernels that take A at any element, chosen for its layout where one that reads vectors would be allowed: A's alignment
        // still has to be what those vectors ask (a move into a packed copy is planned for the declared alignment and refuses
        // an operand below it, whichever kernel it runs).  `linear`: the vectors run along A's first two modes.
        auto vectorsOfA = [&](bool linear) {
            std::vector<int64_t> others;
            for(int d = 1; d < r; ++d)
                if(!linear || d != jB)
                    others.push_back(as[d]);
            return in.elem_bytes * pickVec(in.elem_bytes, cap, linear ? ext[0] * ext[jB] : ext[0], others, in.A, false);
        };
        int        kernel;
        if(tune.kernel == HIPTK_PERM_GROUPED && (tryGrouped(true, true) || tryShared(true)))
            return PermuteStatus::OK;
        const int  full   = 16 / in.elem_bytes;
        const bool runs   = shared && ext[0] >= full && cap >= full; // a 16-byte vector spans two runs at the most
        const int  sq    = (in.elem_bytes == 4 ? TILES4 : TILES2)[0].ti / 2;
        const bool whole = ext[0] % sq == 0 && ext[jB] % sq == 0;
        // strips of 32 rows and more of a tensor that a few hundred workgroups hold: smaller tiles spread it wider (f32
        // 21311 x 57 8.1 us in strips, 4.7 in tiles of 64 x 64, f16 52296 x 56 7.7 and, grouped, 6.0; but
        // f16 66.1684.35 -> (2,0,1), single elements on one side, 7.3 and 8.9)
        const bool smallStrip = (stripJ || stripI) && tune.kernel < 0 && tune.tile < 0 && cap >= full && count <= (1 << 22)
                                && std::min(ext[0], ext[jB]) >= 32 && std::max(ext[0], ext[jB]) >= 64
                                && (in.elem_bytes == 4 || (ext[0] % 2 == 0 && ext[jB] % 2 == 0));
        if(tune.kernel == HIPTK_PERM_GATHER)
            kernel = HIPTK_PERM_GATHER;
        else if(tune.kernel == HIPTK_PERM_RUNS && runs)
            kernel = HIPTK_PERM_RUNS;
        else if(tune.kernel == HIPTK_PERM_STRIP && (stripJ || stripI))
            kernel = HIPTK_PERM_STRIP;
        else if(tune.kernel == HIPTK_PERM_TILED || tune.kernel == HIPTK_PERM_ROWS)
            kernel = shared ? HIPTK_PERM_ROWS : HIPTK_PERM_TILED;
        else if(count <= 16384)
            kernel = HIPTK_PERM_GATHER; // a launch's worth of latency either way
        else if(!shared && count < (1 << 18) && !whole && tune.tile < 0 && tune.gather)
            // Tiles make too few workgroups: f32 238 x 117 6.4 us in tiles, 2.3 here; f16 80 x 3213 8.1 and 3.1; f16
            // 57 x 749 in strips 13.7 and 2.4.  (Extents that the small tiles cover to the last lane: 3.5-3.6 us in those.)
            kernel = HIPTK_PERM_GATHER;
        else if(smallStrip && in.elem_bytes == 4)
        {
            kernel      = HIPTK_PERM_TILED;
            out.a_align = vectorsOfA(stripI);
        }
        else if(smallStrip && tryGrouped(true, false))
        {
            out.a_align = vectorsOfA(stripI);
            return PermuteStatus::OK;
        }
        else if((stripJ && ext[0] >= 64) || (stripI && ext[jB] >= 64))
            kernel = HIPTK_PERM_STRIP;
        else if(shared && tune.tile < 0 && tryShared(false))
            return PermuteStatus::OK;
        else if(shared)
            kernel = ext[0] >= 16 ? HIPTK_PERM_ROWS : HIPTK_PERM_GATHER;
        // (the plain tiles need 16 and more; and up to 2^23 f16 they make too few workgroups, where grouped ones are cut
        // until they make enough: 692 x 464 10.1 us in tiles, 4.2 grouped, 691 x 4279 11.8 and 7.2, 123 x 40061 11.1 and 10.2)
        else if(tune.tile < 0 && tryGrouped(ext[0] < 16 || ext[jB] < 16, false))
            return PermuteStatus::OK;
        else if(tune.tile < 0 && tune.kernel < 0 && in.elem_bytes == 2 && count <= (1 << 23) && (count >= (1 << 18) || !whole) && tryGrouped(true, false))
        {
            out.a_align = vectorsOfA(false);
            return PermuteStatus::OK;
        }
        else
        {
            kernel = (ext[0] >= 16 && ext[jB] >= 16) ? HIPTK_PERM_TILED : HIPTK_PERM_GATHER;
            // blocks transposed in place, which no tile can be put together from: one thread per element reads and writes
            // them from the caches (f16 19.25.23.8.29 -> (1,0,4,2,3) 66 us in tiles, 7.8 here; f32 19.25.230.29 21 and 10)
            const int    order[] = {0, 1, 2};
            const Tile   t       = (in.elem_bytes == 4 ? TILES4 : TILES2)[pickTile(in.elem_bytes, ext[0], ext[jB], order)];
            const double inside  = coverage(ext[0], t.ti) * coverage(ext[jB], t.tj);
            if(tune.kernel < 0 && tune.tile < 0 && inside < 0.15 && kernel == HIPTK_PERM_TILED)
            {
                kernel      = HIPTK_PERM_GATHER;
                out.a_align = vectorsOfA(false);
            }
        }
        out.kernel = kernel;
        if(kernel == HIPTK_PERM_GATHER)
            return PermuteStatus::OK;
        if(kernel == HIPTK_PERM_RUNS)
        {
            out.vec_r = out.vec_w = full;
            return PermuteStatus::OK;
        }

        out.mode_i = 0;
        if(kernel == HIPTK_PERM_STRIP)
        {
            out.mode_j = jB;
            out.tile   = stripJ ? 0 : 1;
            const int64_t        run = ext[0] * ext[jB];
            std::vector<int64_t> linOthers, rowOthers;
            for(int d = 1; d < r; ++d)
            {
                if(d != jB)
                    linOthers.push_back(stripJ ? bs[d] : as[d]);
                if(stripJ || d != jB)
                    rowOthers.push_back(stripJ ? as[d] : bs[d]);
            }
            if(!stripJ)
                rowOthers.push_back(bs[0]);
            if(stripJ)
            {
                out.vec_r = pickVec(in.elem_bytes, cap, ext[0], rowOthers, in.A, false);
                out.vec_w = pickVec(in.elem_bytes, cap, run, linOthers, in.B, false);
            }
            else
            {
                out.vec_r = pickVec(in.elem_bytes, cap, run, linOthers, in.A, false);
                out.vec_w = pickVec(in.elem_bytes, cap, ext[jB], rowOthers, in.B, false);
            }
            return PermuteStatus::OK;
        }
        std::vector<int64_t> aOthers(as.begin() + 1, as.end());
        const int            vr = pickVec(in.elem_bytes, cap, ext[0], aOthers, in.A, false);
        if(kernel == HIPTK_PERM_TILED)
        {
            out.mode_j = jB;
            // (sixteen tiles along j before the next along i: with each die taking neighbouring tiles 0.97 of the time of one)
            out.group = tune.group >= 0 ? tune.group : 16;
            std::vector<int64_t> bOthers;
            for(int d = 0; d < r; ++d)
                if(d != jB)
                    bOthers.push_back(bs[d]);
            out.vec_r         = vr;
            out.vec_w         = pickVec(in.elem_bytes, cap, ext[jB], bOthers, in.B, false);
            const int order[] = {0, 1, 2};
            out.tile          = tune.tile >= 0 && tune.tile <= 3 ? tune.tile : pickTile(in.elem_bytes, ext[0], ext[jB], order);
            // The 64 KiB tile doubles the contiguous run (on both sides for f32: 512 bytes; on A's
            // side for f16), which HBM rewards as long as the tile grid does not lose much more
            // of it at the edges.
            // (and it leaves workgroups enough: f32 5128 x 880 12.2 us in 287 tiles of 64 KiB, 9.1 in small ones, but 729.42.226
            // -> (2,0,1) 14.6 in 504 and 19.3)
            if(tune.tile < 0)
            {
                const Tile*   ts    = in.elem_bytes == 4 ? TILES4 : TILES2;
                const double  cur   = coverage(ext[0], ts[out.tile].ti) * coverage(ext[jB], ts[out.tile].tj);
                const double  big   = coverage(ext[0], ts[3].ti) * coverage(ext[jB], ts[3].tj);
                const int64_t tiles = ((ext[0] + ts[3].ti - 1) / ts[3].ti) * ((ext[jB] + ts[3].tj - 1) / ts[3].tj) * (count / (ext[0] * ext[jB]));
                const double  sq    = coverage(ext[0], ts[0].ti) * coverage(ext[jB], ts[0].tj);
                if(smallStrip)
                    out.tile = 0;
                else if(big >= 0.9 * cur)
                    out.tile = tiles >= 384 || sq < 0.8 * cur ? 3 : 0;
            }
            // Narrow vectors are bound by the number of accesses: 16-byte ones at any element instead (those at the end of a
            // line moved back to end with it), for single f16 and for f32 that is read in less (f16 2712 x 81993 230 -> 218
            // us, 1943.205.637 -> (2,1,0) 460 -> 261, 4459 x 2670 26.0 -> 18.1; f32 2073.32.279 -> (2,1,0) 42.9 -> 37.6).  Not
            // for pairs of f16 (324.350.368 -> (1,2,0) 49 -> 61) nor f32 read whole (164.329.609 -> (1,0,2) 62.8 -> 66.7).
            // Of f16 with pairs on one side and single elements on the other not those written in pairs from the tile of 32
            // columns (75 random shapes 1.25 of the time up to 2^25 elements, 1.49 beyond), nor large matrices with columns of 3000
            // and more read in pairs on tiles of 128 columns (258: 1.07, 178 of them above 1.05) or written in pairs from 128 x 128
            // (38: 1.22); with shorter columns, more modes or fewer elements those take 0.79-0.97, the others 0.61-0.95.
            // (Narrow for the extents' sake: a base off its alignment alone keeps the vectors it admits.)
            const int  er = pickVec(in.elem_bytes, full, ext[0], aOthers, nullptr, false), ew = pickVec(in.elem_bytes, full, ext[jB], bOthers, nullptr, false);
            const bool large  = r == 2 && count > (1 << 25) && ext[jB] >= 3000, square = out.tile == 0;
            const bool single = std::min(er, ew) == 1 && !(ew == 2 && (out.tile == 1 || (large && square))) && !(er == 2 && large && (square || out.tile == 3));
            if(tune.loose || (cap >= full && tune.kernel < 0 && (in.elem_bytes == 2 ? single : er < full)))
            {
                out.loose   = 1;
                out.a_align = std::max(out.a_align, out.vec_r * in.elem_bytes);
                out.vec_r = out.vec_w = full;
            }
        }
        else
        {
            // second tile mode: the one B walks next, so that stores sweep B in order
            int mj = 1;
            for(int d = 1; d < r; ++d)
                if(bs[d] < bs[mj])
                    mj = d;
            out.mode_j = mj;
            std::vector<int64_t> bOthers(bs.begin() + 1, bs.end());
            const int            vw = pickVec(in.elem_bytes, cap, ext[0], bOthers, in.B, false);
            out.vec_r = out.vec_w = std::min(vr, vw);
            const int order[]     = {1, 0, 2};
            out.tile              = tune.tile >= 0 && tune.tile <= 2 ? tune.tile : pickTile(in.elem_bytes, ext[0], ext[mj], order);
            // Vectors of the linear output instead of tiles, from 64-byte runs on (below, f16 24.500.700.8 ->
            // (0,2,1,3): 122.6 us on these tiles, 95.4 linear, 65.0 on shared tiles), where
            //   - the run is no multiple of 16 bytes: f32 21.79.79.20.8.7 -> (0,1,3,4,5,2) 443 -> 203 us, f16
            //     229.60.25.24 -> (0,3,2,1) 22.3 -> 10.5, f16 33.500.700.8 -> (0,2,1,3) 430 -> 178;
            //   - the tiles' lanes mostly fall outside: f32 30.7.61.7.7.65 -> (0,4,2,3,1,5) 468 -> 91 (11 % inside),
            //     f16 40.64.128.256 -> (0,3,2,1) 116 -> 77 (31 %), f16 64.64.128.256 -> (0,2,1,3) 104 -> 96, f32
            //     16.64.128.512 146 -> 130 (50 %; but f32 32.64.128.512, half of a square tile, 198 and 201)
            //   - or a square tile cuts the run into 256 bytes: f32 1140.228.824 -> (0,2,1) 626 -> 298 us, f16 1032.191.1182
            //     320 -> 149 (150 random shapes: 0.45-1.04, mean 0.64).
            // Runs of whole 128-byte lines are what tiles do well.  On large tensors (f32 from 2^24, f16 from 2^27 elements)
            // cut runs of whole lines go linear only where the next runs lie near in A (up to 512 of them at most
            // 1 MiB apart; f32 128.64.128.200 -> (0,2,1,3) 301 -> 271, f16 256.64.128.256 383 -> 352, both sides level for f32
            // up to 2^27): far ones make the linear walk read all over the tensor before it comes back to a run's
            // neighbours, which tiles read together (f32 192.128.2730 -> (0,2,1) 97 us in tiles and 111 linear,
            // 128.16.1024.64 -> (0,3,2,1) 199 and 251).  Likewise half-empty tiles that are long along the run
            // (f32 256 x 16 0.79-0.82 of the tiles' time up to 2^22 elements, 0.85-1.42 from 2^24 on; f16
            // 256.32.1024.32 -> (0,3,2,1) 197 and 240).  Over 400 shapes that this leaves in tiles: linear 0.82-1.42, mean 0.99.
            // Whole runs of full vectors that tiles cover stay in tiles: f32 64.64.64.256 -> (0,3,2,1) 100 against
            // 114, 256.64.128.128 347 and 352; and so do tensors that a launch hides on either (33.40.30 4.0 us in
            // tiles and 2.5 linear, 64.40.30 3.1 and 2.4).
            const bool   f32    = in.elem_bytes == 4;
            const Tile   tt     = (f32 ? TILES4 : TILES2)[out.tile];
            const double inside = coverage(ext[0], tt.ti) * coverage(ext[mj], tt.tj);
            const bool   narrow = out.vec_r < full;
            const bool   big    = count >= (f32 ? 1 << 24 : 1 << 27) && ext[0] * in.elem_bytes % 128 == 0;
            const bool   near   = ext[mj] <= 512 && as[mj] * in.elem_bytes <= (1 << 20);
            const bool   tiled  = out.tile == 1 && big && (f32 || !near); // long tiles: half inside is no loss
            const bool   sparse = inside <= ((f32 && out.tile == 0) || tiled ? 0.45 : 0.55);
            const bool   cut    = out.tile == 0 && ext[0] >= 2 * tt.ti && count >= (1 << 22)
                             && (!big || (count >= (1 << 27) && near));
            if(runs && tune.kernel < 0 && tune.tile < 0 && count >= (1 << 17) && ext[0] * in.elem_bytes >= 64
               && (narrow || sparse || cut))
            {
                out.kernel = HIPTK_PERM_RUNS;
                out.mode_j = 0;
                out.tile   = 0;
                out.vec_r = out.vec_w = full;
            }
        }
        return PermuteStatus::OK;
    }

    PermuteStatus plan_permutation(const PermuteIn& in, const PermuteTuning& tune, hiptk_permute_t& out)
    {
        const PermuteStatus st = pick_kernel(in, tune, out);
        if(st != PermuteStatus::OK)
            return st;
        // Runs of B that do not start at the 64 bytes memory is written in: two tiles each write a part of the lines at
        // their edges, which reach memory whole only if both parts meet in one die's cache.  So neighbouring tiles go to
        // one die (`bands`) and their stores are ordinary ones (`keep`): f32 946.579.437 -> (2,1,0) 762 -> 467 us,
        // 2073.32.279 -> (2,1,0) 94 -> 43, f16 2712 x 81993 390 -> 230.
        int64_t count = 1, runs64 = 1;
        int     jB    = 0;
        for(int d = 0; d < out.rank; ++d)
        {
            count *= out.extent[d];
            if(out.b_stride[d] == 1)
                jB = d;
        }
        for(int d = 0; d < out.rank; ++d)
            if(d != jB && out.b_stride[d] * (int64_t)out.elem_bytes % 64 != 0)
                runs64 = 0;
        // (a matrix, or blocks, transposed in place)
        const bool  inPlace = out.rank >= 2 && jB == 1 && out.b_stride[0] == out.extent[1];
        const Tile* ts      = out.elem_bytes == 4 ? TILES4 : TILES2;
        switch(out.kernel)
        {
        case HIPTK_PERM_TILED:
            // In place the order of the tiles decides less where no two tiles write parts of one line: blocks that one tile holds
            // (f32 36.35.2423 -> (1,0,2) 9.9 us, 11.0 with both), runs of whole 64 bytes in vectors that divide them (44 shapes of
            // 2^24 elements and more 1.03 of the time, up to 1.11) and the f16 tile of 512 columns (1.02, up to 1.26).  Elsewhere
            // sixteen tiles along j without a die to share them lose against one tile (f16 342.799.566 -> (1,0,2) 182 -> 233 us, 1848 x
            // 117198 214 -> 276; with both 130 and 204: 415 shapes 0.81 of the time).
            if(inPlace
               && ((out.extent[0] <= ts[out.tile].ti && out.extent[jB] <= ts[out.tile].tj) || (runs64 && !out.loose)
                   || (out.elem_bytes == 2 && ts[out.tile].ti < 64)))
                break;
            // neighbours on one die also share what they read: 46 random shapes 0.92 of the time, aligned ones among them
            // (f32 1 GiB 379.5 -> 371).  Ordinary stores where the runs are shorter than lines, and on tensors the caches
            // do not hold (up to there they cost 5-10 %: f32 3607 x 590 7.8 -> 8.5, 2307 x 2322 11.8 -> 12.9).
            out.bands = 1;
            out.keep  = !runs64
                       && (ts[out.tile].tj * out.elem_bytes <= 128 || (count >= (1 << 23) && out.vec_w * out.elem_bytes < 16)
                           || count >= (1 << 24) || (out.loose && out.elem_bytes == 2));
            break;
        case HIPTK_PERM_GROUPED:
            // 30 random shapes 0.91 of the time on neighbouring tiles (f32 8.57.15.7.55.66 -> (5,4,2,3,1,0) 490 -> 323, 1.02
            // at the worst), 0.90 with ordinary stores besides
            // (not in place, where such blocks share no line: f16 96.78.191.51 -> (1,0,2,3) 55 us, 63 with both)
            if(inPlace)
                break;
            out.bands = 1;
            out.keep  = !runs64;
            break;
        // (strips and shared tiles with both: 0.98 and 0.96 over 29 shapes, and the choice between two stores costs small
        // ones up to 11 %, f16 45.625.454 -> (1,2,0) 15.5 -> 17.3)
        default: break;
        }
        return PermuteStatus::OK;
    }
}
