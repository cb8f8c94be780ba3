// tile.hpp — one workgroup's share of a temporally blocked pass held in LDS: NS fused
// stream + collide steps of one rectangular tile (grids too small for the column walk of
// multistep.hpp to fill the chip), shared by the single-lattice pass kernel (tile.hip) and
// the batched engine (batch.hip).  See tile.hip for the scheme.
#pragma once

#include <cmath>

#include "common.hpp"
#include "d2q9.hpp"
#include "stepper.hpp"

namespace plbm {

// A tile's region at level 1 holds at most XW columns of H rows; T threads work on it.
// LDS of the shapes in FP64: 41, 73, 78 and 159 of a CU's 160 KB.  The first two are for grids
// that give a CU one tile: its 16 wavefronts then take at most one cell per thread and level
// (64^2 BGK FP64 11 steps, 24 x 24 with 512 / 576 / 1024 threads: 1.00 / 0.95 / 0.95 us per
// step; 128^2 TRT 9 steps 1.05 / 1.02 / 0.97).  Measured and not kept: 24 x 24 with 256, 320 or
// 512 threads (5-15% slower, or within 4%), M with 1024, L with 512 or 768 (3-13% slower),
// 18 x 18, 40 x 36, and 70 x 64 for 4-byte values (5-45% slower than L).
template <int XW_, int H_, int T_, int MEM8_, int MEM4_, int CROWD8_, int CROWD4_>
struct TileShape {
    static constexpr int XW = XW_, H = H_, T = T_;
    // for pick_tile, 8-byte values and smaller ones: cost of moving one cell between memory and
    // LDS in hundredths of a cell's step, and a tile's time in hundredths of its time alone
    // where a CU has several (those of M overlap best)
    static constexpr int MEM8 = MEM8_, MEM4 = MEM4_, CROWD8 = CROWD8_, CROWD4 = CROWD4_;
};
using TileS = TileShape<24, 24, 1024, 107, 120, 114, 119>;
using TileW = TileShape<32, 32, 1024, 100, 115, 105, 103>;
using TileM = TileShape<34, 32, 512, 103, 135, 91, 80>;
using TileL = TileShape<48, 46, 1024, 123, 127, 100, 91>;
constexpr int kTileShapes = 4, kTileM = 2;  // S, W, M, L
constexpr int kMaxTileSteps = 11;  // leaves S tiles of 4 x 4

template <class F>
inline int dispatch_tile_shape(int shape, F &&f) {
    switch (shape) {
    case 0: return f(TileS{});
    case 1: return f(TileW{});
    case kTileM: return f(TileM{});
    default: return f(TileL{});
    }
}

// Most cells a tile of `shape` advances by ns steps: columns, rows.
inline void tile_limits(int shape, int ns, int *w, int *h) {
    dispatch_tile_shape(shape, [&](auto s) {
        using S = decltype(s);
        *w = S::XW - 2 * (ns - 1);
        *h = S::H - 2 * (ns - 1);
        return 0;
    });
}

// RR steps take this many times a BGK or TRT step: memory and launches cost the fewer of them.
inline double tile_heavy(TileKind kind) {
    return kind.model != PLBM_RR ? 1.0 : kind.bytes == 8 ? 1.55 : 1.25;
}
// Work of one tile of w x h cells and ns steps, in steps of a cell (TRT FP64: 0.9 ns): the
// steps of its shrinking levels, the load of its region and the store of its cells, and a ramp.
inline double tile_cell_steps(int ns, int w, int h) {
    double c = 0;
    for (int k = 0; k < ns; ++k) c += double(w + 2 * k) * (h + 2 * k);
    return c;
}
inline double tile_cells_moved(int ns, int w, int h) {
    return double(w + 2 * ns) * (h + 2 * ns) + double(w) * h;
}
inline double tile_work(int shape, TileKind kind, int ns, int w, int h) {
    const int mem = dispatch_tile_shape(shape, [&](auto s) {
        return kind.bytes == 8 ? decltype(s)::MEM8 : decltype(s)::MEM4;
    });
    return tile_cell_steps(ns, w, h) +
           (0.01 * mem * tile_cells_moved(ns, w, h) + 850) / tile_heavy(kind);
}
// Time of the busiest CU when `tiles` tiles are shared out, in units of one tile's work.
inline double tile_rounds(int shape, TileKind kind, double tiles) {
    if (tiles <= kComputeUnits) return 1;
    const int crowd = dispatch_tile_shape(shape, [&](auto s) {
        return kind.bytes == 8 ? decltype(s)::CROWD8 : decltype(s)::CROWD4;
    });
    return 0.01 * crowd * std::ceil(tiles / kComputeUnits);
}
// A launch, in the same unit.
inline double tile_launch_work(TileKind kind) {
    return (kind.bytes == 8 ? 2000 : 3400) / tile_heavy(kind);
}

// The shape and depth (in [ns_min, ns_max]) that cost the least per step on an nx x ny
// grid; returns the cost of a step.  The constants above are fitted to every shape and depth
// to 16 on 16 grids of 32^2 to 1280^2 and three collisions: the choice, free or at a given
// depth, is on average 0.2% slower than the fastest measured, at most 4%.  The depth that
// leaves just 256 tiles mostly wins, e.g. TRT FP64 640^2 4 steps of L, 5.3 -> 4.1 us per step,
// 400^2 11 steps of L, 2.5 -> 2.0.
double pick_tile(int nx, int ny, TileKind kind, int ns_min, int ns_max, int *shape, int *ns);

// The depth that makes nsteps >= 2 steps, spread evenly over their passes, cost the least.
int tile_depth(int nx, int ny, TileKind kind, int nsteps);

// Column / row boundary j of n cells cut into m nearly equal parts, long and short ones mixed
// (all longer ones first made the last CUs to finish later: 1001 x 777 RR passes 4%, batches
// 7%).  In 32 bits where they suffice: a workgroup's four boundaries by 64-bit divisions took
// 600 scalar instructions, 2-3% of a pass of a small grid (64^2 BGK 1.20 -> 1.16 us per step).
__host__ __device__ inline int part_start(int n, int m, int j) {
    if (n < 65536 && m < 65536) return (int)((unsigned)n * (unsigned)j / (unsigned)m);  // j <= m
    return (int)((long long)n * j / m);
}

__host__ __device__ constexpr int opposite(int q) {
    return q == 0 ? 0 : (q < 5 ? (q + 1) % 4 + 1 : (q - 3) % 4 + 5);
}
static_assert(opposite(1) == 3 && opposite(2) == 4 && opposite(3) == 1 && opposite(4) == 2 &&
                  opposite(5) == 7 && opposite(6) == 8 && opposite(7) == 5 && opposite(8) == 6,
              "opposite directions");

__device__ __forceinline__ int wrap_index(int v, int n) {
    if (v < 0 || v >= n) {
        v %= n;
        if (v < 0) v += n;
    }
    return v;
}

// One cell's collision in a tile.  WIDE (FP32 storage, BGK): in FP64 on the FP32 populations,
// rounded once.  Where a tile replaces the column walk, whose FMAs the compiler places
// differently at every level, the FP32 BGK arithmetic of single steps was 5-12% further off
// the FP64 run (velocity after 300-600 steps at nu = 0.03: 9.3e-7 to 1.7e-6 against 8.1e-7 to
// 1.5e-6); in FP64 it is 4.2e-8 to 4.6e-8.  Of the other FP32 collisions RR has the walk's
// bits and TRT its error.
template <int MODEL, int ST, bool WIDE>
__device__ __forceinline__ void collide_tile(typename Traits<ST>::R (&f)[9], const StepArgs &a) {
    if constexpr (WIDE) {
        double g[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) g[q] = double(f[q]);
        collide_bgk_shifted<double>(g, a.omega);
#pragma unroll
        for (int q = 0; q < 9; ++q) f[q] = float(g[q]);
    } else {
        collide_cell<MODEL, ST>(f, a);
    }
}
// Whether passes of this storage and model are WIDE where they do not stand for single steps.
constexpr bool tile_wide(int storage, int model) {
    return storage == PLBM_F32S && (model == PLBM_BGK || model == PLBM_BGK_SPLIT);
}

// The calling workgroup (SHAPE::T threads) advances cells [x0, x0 + w) x [y0, y0 + h) of
// the grid described by `a` ns >= 1 steps, a.src -> a.dst, and, when a.lag is set (ns >= 2),
// stores the state one step before there.  w + 2 (ns - 1) <= XW, h + 2 (ns - 1) <= H.
// KEEP: every level is stored (StepArgs::level_stride).
//
// LDS holds one copy of the region's populations, updated in place.  A step pulls f_q(x)
// from cell x - c_q, so writing the result where it was read from (A: the value of the
// opposite direction goes to (x - c_q, q), where the next step's pull would send it) makes
// the step after it a purely local one (B: direction p is read from (x, opposite(p)) and
// written back to (x, p)).  Every LDS word is read and written by the same thread in a
// step, so that one barrier per step suffices, any number of cells per thread works, and
// half the LDS of a ping-pong pair holds the tile.
template <int MODEL, int ST, class SHAPE, bool WIDE = false, bool KEEP = false>
__device__ __forceinline__ void tile_steps(const StepArgs &a, int ns, int x0, int w, int y0,
                                           int h) {
    using T = typename Traits<ST>::T;
    using R = typename Traits<ST>::R;
    constexpr int H = SHAPE::H, NT = SHAPE::T;
    __shared__ R mem[SHAPE::XW * 9 * H];  // (lx, q, ly)
    const T *__restrict__ s = static_cast<const T *>(a.src);
    T *__restrict__ d = static_cast<T *>(a.dst);
    T *__restrict__ lag = static_cast<T *>(a.lag);
    const int nx = a.nx, ny = a.ny, halo = ns - 1;
    const size_t L = (size_t)a.ldd;
    // FP16 storage with a.round_levels: every level rounded as a single step's store and the
    // next one's load round it
    auto settle = [&](R(&f)[9]) __attribute__((always_inline)) {
        if constexpr (ST == PLBM_F16S) {
            if (a.round_levels)
#pragma unroll
                for (int q = 0; q < 9; ++q) f[q] = R(T(f[q] * a.scale)) * a.inv_scale;
        }
    };
    auto store = [&](T *to, int lx, int ly, const R(&f)[9]) __attribute__((always_inline)) {
        const int ox = lx - halo, oy = ly - halo;
        if (ox < 0 || ox >= w || oy < 0 || oy >= h) return;
        T *p = to + (size_t)(x0 + ox) * a.cs + (y0 + oy);
#pragma unroll
        for (int q = 0; q < 9; ++q) store_pop<ST, false>(p + q * L, f[q], a.scale);
    };

    // level 1 from global memory, over the whole region
    {
        const int w1 = w + 2 * halo, h1 = h + 2 * halo, n = w1 * h1;
        const float rh = 1.0f / float(h1);
        for (int i = threadIdx.x; i < n; i += NT) {
            const int lx = int((float(i) + 0.5f) * rh), ly = i - lx * h1;
            const int x = wrap_index(x0 - halo + lx, nx), y = wrap_index(y0 - halo + ly, ny);
            const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
            const int ym = y == 0 ? ny - 1 : y - 1, yp = y == ny - 1 ? 0 : y + 1;
            const size_t c0 = (size_t)x * a.cs, cm = (size_t)xm * a.cs, cp = (size_t)xp * a.cs;
            const float is = a.inv_scale;
            R f[9];
            f[0] = load_pop<ST>(s + c0 + 0 * L + y, is);
            f[1] = load_pop<ST>(s + cm + 1 * L + y, is);
            f[2] = load_pop<ST>(s + c0 + 2 * L + ym, is);
            f[3] = load_pop<ST>(s + cp + 3 * L + y, is);
            f[4] = load_pop<ST>(s + c0 + 4 * L + yp, is);
            f[5] = load_pop<ST>(s + cm + 5 * L + ym, is);
            f[6] = load_pop<ST>(s + cp + 6 * L + ym, is);
            f[7] = load_pop<ST>(s + cp + 7 * L + yp, is);
            f[8] = load_pop<ST>(s + cm + 8 * L + yp, is);
            collide_tile<MODEL, ST, WIDE>(f, a);
            if (halo == 0) {  // one step: nothing to hand on
                store(d, lx, ly, f);
                continue;
            }
            settle(f);
            R *m = mem + lx * 9 * H + ly;
#pragma unroll
            for (int q = 0; q < 9; ++q) m[q * H] = f[q];
            if constexpr (KEEP) store(d, lx, ly, f);
            else if (halo == 1 && lag != nullptr) store(lag, lx, ly, f);
        }
    }
    // levels 2 .. ns, each one cell smaller on every side: the even ones A, the odd ones B
    auto level = [&](int k, auto odd, auto last) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd)::value, LAST = decltype(last)::value;
        const int hk = h + 2 * (ns - k), n = (w + 2 * (ns - k)) * hk;
        const float rh = 1.0f / float(hk);
        for (int i = threadIdx.x; i < n; i += NT) {
            const int ix = int((float(i) + 0.5f) * rh);
            const int lx = ix + k - 1, ly = i - ix * hk + k - 1;
            R *m = mem + lx * 9 * H + ly;
            R f[9];
#pragma unroll
            for (int q = 0; q < 9; ++q)
                f[q] = ODD ? m[opposite(q) * H] : m[(q - 9 * cx(q)) * H - cy(q)];
            collide_tile<MODEL, ST, WIDE>(f, a);
            if constexpr (LAST) {
                store(KEEP ? d + (size_t)(k - 1) * a.level_stride : d, lx, ly, f);
            } else {
                settle(f);
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if constexpr (ODD) m[q * H] = f[q];
                    else m[(q - 9 * cx(q)) * H - cy(q)] = f[opposite(q)];
                if constexpr (KEEP) store(d + (size_t)(k - 1) * a.level_stride, lx, ly, f);
                else if (k == halo && lag != nullptr) store(lag, lx, ly, f);
            }
        }
    };
    if (halo == 0) return;
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    for (int k = 2; k < ns; ++k) {
        __syncthreads();
        if (k & 1) level(k, yes, no);
        else level(k, no, no);
    }
    __syncthreads();
    if (ns & 1) level(ns, yes, yes);
    else level(ns, no, yes);
}

}  // namespace plbm
