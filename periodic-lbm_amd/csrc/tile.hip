// tile.hip — temporally blocked passes of small and medium grids, held in LDS.
//
// The column walk of multistep.hip needs a long walk per wavefront and about a thousand
// wavefronts: below about 1000^2 its start-up columns (2 NS per segment) and idle SIMDs cost
// more than the steps, and below about 500^2 single steps, one launch of 2.5-3.5 us each,
// were faster.  Here a workgroup advances one rectangular tile ns steps in LDS (tile.hpp):
// level 1 is pulled from global memory over the tile and its halo of ns - 1 cells on each
// side, each further level is one cell smaller on every side, and the last is stored.  What
// bounds it: a CU's VALU issue plus the LDS traffic that does not overlap it (512^2 TRT FP64,
// 8 steps: 58% of the issue slots of the busy CUs, 38% LDS active, a fifth of that bank
// conflicts where a wavefront crosses a column), the launch for the smallest grids.  Two
// cells per thread and iteration, to overlap one's LDS reads with the other's collision,
// measured 3-20% slower.
//
// us per step, single steps / column walk of 8 / tiles: 64^2 BGK FP64 3.4 / 5.5 / 0.9;
// 192^2 TRT FP64 3.6 / 4.9 / 1.2; 512^2 TRT FP64 8.3 / 5.0 / 2.3, FP32 4.3 / 3.5 / 1.6;
// 1001 x 777 RR FP64 23.8 / 24.5 / 10.1; 1024^2 TRT FP64 29 / 10.0 / 8.4, FP32 16.4 / 5.8 /
// 4.2.  Tiles of up to 11 steps in four shapes instead of up to 8 in three, 512^2 and larger
// ones mostly the same: 64^2 BGK FP64 1.08 -> 0.90, 128^2 TRT FP64 1.15 -> 0.97, 320^2 RR
// FP64 2.43 -> 2.23, 400^2 TRT FP64 2.50 -> 1.99, 640^2 TRT FP64 5.3 -> 4.1, FP32 3.1 -> 2.1.
//
// Per-cell arithmetic is collide_cell, as everywhere: FP64 results equal single steps bit
// for bit, and the shifted FP64 / FP32 storages did on every case compared (but see
// collide_tile for FP32 BGK).
#include "tile.hpp"

namespace plbm {

template <int MODEL, int ST, class SHAPE, bool WIDE, bool KEEP = false>
__global__ void __launch_bounds__(SHAPE::T) __attribute__((amdgpu_waves_per_eu(4)))
    k_tile(StepArgs a, int ns, int nbx, int nby) {
    const int b = xcd_remap(blockIdx.x, gridDim.x);  // neighbouring tiles share an L2
    const int by = b % nby, bx = b / nby;
    const int x0 = part_start(a.nx, nbx, bx), x1 = part_start(a.nx, nbx, bx + 1);
    const int y0 = part_start(a.ny, nby, by), y1 = part_start(a.ny, nby, by + 1);
    tile_steps<MODEL, ST, SHAPE, WIDE, KEEP>(a, ns, x0, x1 - x0, y0, y1 - y0);
}

double pick_tile(int nx, int ny, TileKind kind, int ns_min, int ns_max, int *shape, int *ns) {
    double best = 1e300;
    for (int n = ns_min; n <= ns_max; ++n)
        for (int s = 0; s < kTileShapes; ++s) {
            int w, h;
            tile_limits(s, n, &w, &h);
            const long long nbx = (nx + w - 1) / w, nby = (ny + h - 1) / h;
            w = (int)((nx + nbx - 1) / nbx);
            h = (int)((ny + nby - 1) / nby);
            const double c = (tile_launch_work(kind) + tile_rounds(s, kind, double(nbx * nby)) *
                                                           tile_work(s, kind, n, w, h)) /
                             n;
            if (c < best) {
                best = c;
                *shape = s;
                *ns = n;
            }
        }
    return best;
}

int tile_depth(int nx, int ny, TileKind kind, int nsteps) {
    double cost[kMaxTileSteps + 1] = {}, least = 1e300;
    int best = 2;
    for (int n = 1; n <= kMaxTileSteps; ++n) {
        int shape, ns;
        cost[n] = n * pick_tile(nx, ny, kind, n, n, &shape, &ns);
        const int passes = (nsteps + n - 1) / n, d = nsteps / passes, deeper = nsteps % passes;
        const double c = (passes - deeper) * cost[d] + (deeper ? deeper * cost[d + 1] : 0.0);
        if (n >= 2 && c < least) {
            least = c;
            best = n;
        }
    }
    return best;
}

TileKind tile_kind(const plbm_lattice *h, int model) {
    return {(int)storage_bytes(h->storage), model};
}

// Grids up to this many cells take tiles: about where the column walk catches up.  us per
// step of 96 steps at both sides' automatic depths, column walk / tiles:
//         FP64                                   FP32                    FP16
//   BGK   1000^2 10.4/9.2, 1150^2 12.8/12.4,     (below)                 1450^2 8.3/8.1,
//         1300^2 14.4/16.6                                               1600^2 9.3/9.9
//   TRT   800^2 6.8/5.8, 900^2 7.4/7.8,          1150^2 5.5/5.2,         1150^2 5.6/5.2,
//         1150^2 10.3/11.4                       1300^2 6.2/7.1          1300^2 6.4/6.9
//   RR    1150^2 18.2/16.4, 1300^2 22.5/20.8,    1600^2 14.6/13.0,       1450^2 12.9/12.1,
//         1450^2 26.1/28.4                       2048^2 21.7/22.4        1800^2 18.1/17.7
// FP32 BGK in FP64 arithmetic (collide_tile): 640^2 4.9/3.9, 800^2 5.3/4.9, 1001 x 777 5.8/5.2,
// 1024^2 5.9/6.0.
bool tile_cells(int storage, int model, long long cells) {
    const int bytes = (int)storage_bytes(storage);
    const auto pick = [&](long long f64, long long f32, long long f16) {
        return cells <= (bytes == 8 ? f64 : bytes == 4 ? f32 : f16);
    };
    if (model == PLBM_TRT) return pick(750000, 1400000, 1400000);
    if (model == PLBM_RR) return pick(1800000, 3300000, 2600000);
    return pick(1400000, 850000, 2200000);
}

// Long grids of few columns are mostly halo as tiles, and give the column walk a wavefront per
// band: us per step in runs of 4 / 40 steps, walks and tiles: 1 x 60000 BGK FP64 6.8 / 7.1, 9.3 /
// 6.4, TRT FP32 4.9 / 2.9, 6.2 / 3.4, 2 x 200000 FP64 12.1 / 18.3, 25 / 22, 8 x 60000 BGK FP32
// 7.9 / 5.2, 9.0 / 6.1; but 1 x 25000 BGK FP64 5.9 / 3.8, 5.5 / 3.3, 6 x 60000 10.0 / 10.1, 11.2 /
// 8.3.  A caller who chose the column walk's segments (plbm_set_pass_segments) keeps it.
bool tile_grid(const plbm_lattice *h, int model) {
    const bool slender = h->ny > 32768 && h->nx <= (h->storage == PLBM_F32S ? 8 : 4);
    return h->pass_segs == 0 && !slender &&
           tile_cells(h->storage, model, (long long)h->nx * h->ny);
}

static StepArgs tile_args(const plbm_lattice *h, const void *src, void *dst, void *lag) {
    StepArgs a{};
    a.src = src;
    a.dst = dst;
    a.lag = lag;
    a.nx = h->nx;
    a.ny = h->ny;
    a.ldd = h->ldd;
    a.cs = (size_t)9 * h->ldd;
    a.omega = h->omega;
    a.lambda_odd = h->lambda_odd;
    a.omega_f = float(h->omega);
    a.lambda_odd_f = float(h->lambda_odd);
    a.scale = float(h->scale);
    a.inv_scale = float(1.0 / h->scale);
    return a;
}

int launch_tile(plbm_lattice *h, int model, int ns, const void *src, void *dst, void *lag,
                bool as_single) {
    StepArgs a = tile_args(h, src, dst, lag);
    a.round_levels = as_single && h->storage == PLBM_F16S;
    int shape = 0, wx, wy;
    pick_tile(h->nx, h->ny, tile_kind(h, model), ns, ns, &shape, &ns);
    tile_limits(shape, ns, &wx, &wy);
    const int nbx = (h->nx + wx - 1) / wx, nby = (h->ny + wy - 1) / wy;
    return dispatch_model(model, [&](auto M) {
        return dispatch_storage(h->storage, [&](auto S) {
            return dispatch_tile_shape(shape, [&](auto sh) {
                constexpr int MM = decltype(M)::value, SS = decltype(S)::value;
                using SH = decltype(sh);
                auto go = [&](auto wide) {
                    hipLaunchKernelGGL((k_tile<MM, SS, SH, decltype(wide)::value>),
                                       dim3((unsigned)(nbx * nby)), dim3(SH::T), 0, h->stream, a,
                                       ns, nbx, nby);
                };
                if (tile_wide(SS, MM) && !as_single)
                    go(std::integral_constant<bool, tile_wide(SS, MM)>{});
                else
                    go(std::false_type{});
                PLBM_HIP(hipGetLastError());
                return PLBM_OK;
            });
        });
    });
}

int launch_tile_levels(plbm_lattice *h, int ns, const void *src, void *dst) {
    StepArgs a = tile_args(h, src, dst, nullptr);
    a.level_stride = h->elems;
    int shape = 0, wx, wy;
    pick_tile(h->nx, h->ny, tile_kind(h, PLBM_BGK), ns, ns, &shape, &ns);
    tile_limits(shape, ns, &wx, &wy);
    const int nbx = (h->nx + wx - 1) / wx, nby = (h->ny + wy - 1) / wy;
    return dispatch_storage(h->storage, [&](auto S) {
        constexpr int SS = decltype(S)::value;
        if constexpr (SS == PLBM_F16S) {
            set_error("passes that keep every level need FP64 or FP32 storage");
            return PLBM_ERR_ARG;
        } else {
            return dispatch_tile_shape(shape, [&](auto sh) {
                using SH = decltype(sh);
                hipLaunchKernelGGL((k_tile<PLBM_BGK, SS, SH, false, true>),
                                   dim3((unsigned)(nbx * nby)), dim3(SH::T), 0, h->stream, a, ns,
                                   nbx, nby);
                PLBM_HIP(hipGetLastError());
                return PLBM_OK;
            });
        }
    });
}

}  // namespace plbm
