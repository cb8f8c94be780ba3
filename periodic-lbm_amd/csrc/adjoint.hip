// adjoint.hip — discrete adjoint of the BGK stream-collide step with checkpointing.
//
// Forward map (one step n):  g^n = S f^n (pull streaming),  f^{n+1} = C(g^n) =
// (1-omega) g^n + omega feq(rho(g^n), u(g^n)).  Initial state f^0 = feq(rho0, u0); loss
// L = 1/2 sum_cells |u(f^N) - u*|^2 with u = j/rho.
//
// Reverse sweep: lambda^N = dL/df^N; for n = N-1 .. 0
//   mu      = J_C(g^n)^T lambda^{n+1}          (collision Jacobian at the pre-collision state)
//   lambda^n_q(x - c_q) = mu_q(x)              (S^T: push streaming)
//   dL/domega += sum_cells sum_q lambda^{n+1}_q (feq_q(g^n) - g^n_q)
// and dL/du0, dL/drho0 = (d feq / d(rho, u))^T lambda^0.
//
// Memory: states are checkpointed every K steps during the forward sweep, which leaves the
// last K-step segment's states in a segment buffer; the reverse sweep recomputes each earlier
// segment into it from its checkpoint before it runs the K reverse steps (a further backward
// call the last one too).  Forward cost about 2N - K steps, reverse N steps.
//
// All three run in LDS tiles of several steps: the forward from checkpoint to checkpoint
// (tile.hip), the recomputation storing every level on its way, the reverse sweep in
// k_adj_tile.  512^2 FP64, per step: forward 8.9 us in single steps -> 3.1, recomputation
// 8.9 -> 4.0 (its writes at 4.7 TB/s), reverse 12.8 -> 7.0.
//
// For BGK with rho = sum g, u = sum c g / rho, feq_i = w_i rho (1 + P_i),
// P_i = 3 c_i.u + 4.5 (c_i.u)^2 - 1.5 u.u:
//   d feq_i / d rho = w_i (1 + P_i),  d feq_i / d u_a = w_i rho (3 c_ia + 9 (c_i.u) c_ia - 3 u_a)
//   d rho / d g_j = 1,  d u_a / d g_j = (c_ja - u_a) / rho
//   mu_j = (1-omega) lambda_j + omega (A + sum_a B_a (c_ja - u_a) / rho),
//   A = sum_i lambda_i w_i (1 + P_i),  B_a = sum_i lambda_i d feq_i / d u_a.
#include <algorithm>
#include <cmath>
#include <string>
#include <utility>
#include <vector>

#include "common.hpp"
#include "d2q9.hpp"
#include "stepper.hpp"
#include "tile.hpp"

namespace plbm {

constexpr int kAdjBlocks = 2048;  // reduction partial slots (fixed => deterministic)

// Macros of one stored cell (pulled or not) from its populations g (deviations
// g_q = f_q - w_q for the shifted storages), in the adjoint's FP64 arithmetic.
template <bool SHIFTED>
__device__ __forceinline__ void cell_state(const double gs[9], double &rho, double &ux,
                                           double &uy, double &drho) {
    double d, jx, jy;
    moments_shifted<double>(gs, d, jx, jy);  // plain sums: valid for shifted and unshifted
    if constexpr (SHIFTED) {
        drho = d;
        rho = 1.0 + d;
    } else {
        rho = d;
        drho = d - 1.0;
    }
    ux = jx / rho;
    uy = jy / rho;
}

// The adjoint state lambda, mu and the omega sensitivity are FP64 for every storage: the
// forward states of FP32 storage convert to FP64 exactly, so the reverse sweep is the
// exact adjoint of the FP64 step evaluated along the FP32 trajectory, and its own
// rounding (500 reverse steps of FP32 would add about 1e-5 relative to the gradient)
// drops out.

// Index of element q at x + c_q, periodic.
__device__ __forceinline__ size_t neighbour(int x, int y, int q, int nx, int ny, int ldd) {
    const int xq = x + cx(q), yq = y + cy(q);
    return pop_index(q, xq < 0 ? nx - 1 : xq == nx ? 0 : xq, yq < 0 ? ny - 1 : yq == ny ? 0 : yq,
                     ldd);
}

// lambda^N, stored as the mu that S^T would make it from, and the loss of the final state.
template <int ST>
__global__ void __launch_bounds__(256)
    k_adj_final(const void *fN, int nx, int ny, int ldd, float inv_scale, const double *uxt,
                const double *uyt, double *mu, double *partials) {
    using T = typename Traits<ST>::T;
    __shared__ double sh[256];
    double acc = 0.0;
    const size_t n = (size_t)nx * ny;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i / ny), y = (int)(i % ny);
        const T *s = static_cast<const T *>(fN);
        const size_t c = pop_index(0, x, y, ldd);
        double g[9];
#pragma unroll
        for (int q = 0; q < 9; ++q)
            g[q] = double(load_pop<ST>(s + c + (size_t)q * ldd, inv_scale));
        double rho, ux, uy, drho;
        cell_state<Traits<ST>::shifted>(g, rho, ux, uy, drho);
        const double ex = ux - uxt[i], ey = uy - uyt[i];
        acc += 0.5 * (ex * ex + ey * ey);
        const double inv = 1.0 / rho;
#pragma unroll
        for (int q = 0; q < 9; ++q)
            mu[neighbour(x, y, q, nx, ny, ldd)] = (ex * (cx(q) - ux) + ey * (cy(q) - uy)) * inv;
    }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = sh[0];
}

// One cell's reverse step: g = g^n, lam = lambda^{n+1} -> mu, and the cell's omega sensitivity
// sum_q lambda_q (feq_q - g_q).  The sums over directions are those of six moments of
// w_q lambda_q, and rho cancels from B_a / rho:
//   A - m = 3 u.m1 + 4.5 u.m2.u - 1.5 u.u m,  B_a / rho = 3 m1_a + 9 (m2.u)_a - 3 u_a m,
//   m = sum w_q lambda_q, m1_a = sum w_q lambda_q c_qa, m2_ab = sum w_q lambda_q c_qa c_qb,
//   sum_q lambda_q feq_q = rho A  (in deviation form drho m + rho (A - m)),
// a third of the operations of the sums written out.  FMAs are written where they are meant,
// so that a cell's result does not depend on the kernel or level that computes it.
template <bool SHIFTED>
__device__ __forceinline__ double adj_cell(const double (&g)[9], const double (&lam)[9],
                                           double omega, double (&mu)[9]) {
#pragma clang fp contract(off)
    const auto fma = [](double p, double q, double r) { return __builtin_fma(p, q, r); };
    double d, jx, jy;
    moments_shifted<double>(g, d, jx, jy);
    const double rho = SHIFTED ? 1.0 + d : d, drho = SHIFTED ? d : d - 1.0;
    const double inv = 1.0 / rho, ux = jx * inv, uy = jy * inv;
    constexpr double w0 = wq(0), w1 = wq(1), w5 = wq(5);
    const double s13 = lam[1] + lam[3], d13 = lam[1] - lam[3];
    const double s24 = lam[2] + lam[4], d24 = lam[2] - lam[4];
    const double s57 = lam[5] + lam[7], d57 = lam[5] - lam[7];
    const double s68 = lam[6] + lam[8], d68 = lam[6] - lam[8];
    const double wd = w5 * (s57 + s68);
    const double m = fma(w0, lam[0], fma(w1, s13 + s24, wd));
    const double mx = fma(w1, d13, w5 * (d57 - d68)), my = fma(w1, d24, w5 * (d57 + d68));
    const double mxx = fma(w1, s13, wd), myy = fma(w1, s24, wd), mxy = w5 * (s57 - s68);
    const double tx = fma(ux, mxx, uy * mxy), ty = fma(ux, mxy, uy * myy);
    const double u2 = fma(ux, ux, uy * uy);
    const double am = fma(3.0, fma(ux, mx, uy * my),
                          fma(4.5, fma(ux, tx, uy * ty), -1.5 * u2 * m));  // A - m
    const double m3 = -3.0 * m;
    const double bx = fma(3.0, mx, fma(9.0, tx, ux * m3));  // B_a / rho
    const double by = fma(3.0, my, fma(9.0, ty, uy * m3));
    const double kx = omega * bx, ky = omega * by, rest = 1.0 - omega;
    const double k0 = fma(omega, m + am, -fma(kx, ux, ky * uy));
    const double kxp = k0 + kx, kxm = k0 - kx;
    mu[0] = fma(rest, lam[0], k0);
    mu[1] = fma(rest, lam[1], kxp);
    mu[2] = fma(rest, lam[2], k0 + ky);
    mu[3] = fma(rest, lam[3], kxm);
    mu[4] = fma(rest, lam[4], k0 - ky);
    mu[5] = fma(rest, lam[5], kxp + ky);
    mu[6] = fma(rest, lam[6], kxm + ky);
    mu[7] = fma(rest, lam[7], kxm - ky);
    mu[8] = fma(rest, lam[8], kxp - ky);
    double sg = 0.0;
#pragma unroll
    for (int q = 0; q < 9; ++q) sg = fma(lam[q], SHIFTED ? g[q] : g[q] - wq(q), sg);
    return fma(drho, m, fma(rho, am, -sg));
}

// Sum of many terms in two doubles (Knuth's two-sum): its error is of the order of the square
// of a double's rounding, so that the total does not depend on how the steps are split into
// passes and the grid into tiles.
struct Sum2 {
    double hi, lo;
    __device__ __forceinline__ void add(double d) {
#pragma clang fp contract(off)
        const double s = hi + d, b = s - hi;
        lo += (hi - (s - b)) + (d - b);
        hi = s;
    }
    __device__ __forceinline__ void add(const Sum2 &o) {
        add(o.hi);
        lo += o.lo;
    }
    // an infinite sum's error term is NaN
    __device__ __forceinline__ double value() const { return isfinite(hi) ? hi + lo : hi; }
};
// Sum over the calling wavefront.
__device__ __forceinline__ Sum2 wave_sum(Sum2 v) {
#pragma unroll
    for (int st = 32; st > 0; st >>= 1) v.add({__shfl_xor(v.hi, st), __shfl_xor(v.lo, st)});
    return v;
}
// Sum over the calling workgroup of NT threads, valid in thread 0; sh holds NT / 64 values.
template <int NT>
__device__ __forceinline__ Sum2 block_sum(Sum2 v, Sum2 *sh) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < NT / 64; ++i) v.add(sh[i]);
    return v;
}

// ns reverse steps of one tile held in LDS, in place as tile_steps holds the forward ones
// (tile.hpp), with every direction turned round: the adjoint state in memory is mu, before
// S^T, so that level 1 pulls lambda_q(x) = mu_q(x + c_q) over the tile and its halo of ns - 1
// cells; an even level gathers from (x + c_q, q) and leaves mu_p where the opposite direction
// was read, an odd one reads (x, opposite(p)) and writes (x, p).  Level l takes g from state
// top - (l - 1) stride, the last from `last`.  The omega sensitivity of the tile's own cells is
// added to the wavefront's partial sum (a sum over the workgroup per pass took 3-4 us; partial
// sums of the threads took 142 MB beside states of 29 MB at 1 x 400000, and their traffic: 512^2,
// 500 steps 6.55 -> 6.50 ms).
//
// Bound by its reads of the states, 1.5 times the tile's own with the halo: at 512^2 4.5 TB/s
// from beyond the L2s, with 42% of the issue slots used.  The whole backward call, 500 steps at
// 512^2, ms, in tiles S / M / L of 4 steps 6.7 / 6.5 / 6.7, of 8 steps 7.7 / 6.2 / 5.4 (L: one
// tile per CU); 100 steps at 1024^2 5.8 - 6.2 from 4 steps on: the forward's choice of shape and
// depth serves.  Loading a thread's next cell ahead, across the barriers, changed nothing (126
// instead of 98 registers), nor did 32-bit offsets in FP64 (FP32 storage 4.4 -> 4.0 ms).
template <int ST>
struct AdjArgs {
    using T = typename Traits<ST>::T;
    const T *top, *last;
    size_t stride, cs;
    const double *mu_in;
    double *mu_out;
    Sum2 *partials;
    int nx, ny, ldd;
    double omega;
    float inv_scale;
};
template <int ST, class SHAPE, bool FAR>
__global__ void __launch_bounds__(SHAPE::T) __attribute__((amdgpu_waves_per_eu(4)))
    k_adj_tile(AdjArgs<ST> a, int ns, int nbx, int nby) {
    using T = typename Traits<ST>::T;
    using Offset = std::conditional_t<FAR, size_t, uint32_t>;  // bytes
    constexpr int H = SHAPE::H, NT = SHAPE::T;
    __shared__ double mem[SHAPE::XW * 9 * H];  // (lx, q, ly)
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int by = b % nby, bx = b / nby;
    const int x0 = part_start(a.nx, nbx, bx), w = part_start(a.nx, nbx, bx + 1) - x0;
    const int y0 = part_start(a.ny, nby, by), h = part_start(a.ny, nby, by + 1) - y0;
    const int nx = a.nx, ny = a.ny, halo = ns - 1;
    const size_t L = (size_t)a.ldd;
    const Offset cs = (Offset)(a.cs * sizeof(T));  // bytes of a column
    // Cell i of level k: in the tile's region, and its offsets and its neighbours' in a state.
    struct Cell {
        int lx, ly;
        Offset c0, cm, cp, r0, rm, rp;
    };
    auto cell = [&](int k, int i, int hk, float rh) __attribute__((always_inline)) {
        const int ix = int((float(i) + 0.5f) * rh);
        Cell c;
        c.lx = ix + k - 1;
        c.ly = i - ix * hk + k - 1;
        const int x = wrap_index(x0 + c.lx - halo, nx), y = wrap_index(y0 + c.ly - halo, ny);
        c.c0 = FAR ? (Offset)x * cs : (Offset)__umul24(x, (uint32_t)cs);
        c.r0 = (Offset)y * sizeof(T);
        const Offset xe = (Offset)(nx - 1) * cs, ye = (Offset)(ny - 1) * sizeof(T);
        c.cm = x == 0 ? c.c0 + xe : c.c0 - cs;
        c.cp = x == nx - 1 ? c.c0 - xe : c.c0 + cs;
        c.rm = y == 0 ? c.r0 + ye : c.r0 - (Offset)sizeof(T);
        c.rp = y == ny - 1 ? c.r0 - ye : c.r0 + (Offset)sizeof(T);
        return c;
    };
    // q's population at x - c_q (S = 1) or x + c_q (-1)
    auto from = [&](const Cell &c, int q, int S) __attribute__((always_inline)) {
        const int dx = S * cx(q), dy = S * cy(q);
        return (dx > 0 ? c.cm : dx < 0 ? c.cp : c.c0) + (dy > 0 ? c.rm : dy < 0 ? c.rp : c.r0);
    };
    auto mu_at = [&](auto *p, int q, Offset o) __attribute__((always_inline)) {
        constexpr Offset wide = sizeof(double) / sizeof(T);
        using C = std::conditional_t<std::is_const_v<std::remove_pointer_t<decltype(p)>>,
                                     const char, char>;
        return reinterpret_cast<decltype(p)>(reinterpret_cast<C *>(p + q * L) + wide * o);
    };
    Sum2 *mine = a.partials + (size_t)blockIdx.x * (NT / 64) + (threadIdx.x >> 6);
    const bool first_lane = (threadIdx.x & 63) == 0;
    Sum2 sum = first_lane ? *mine : Sum2{0.0, 0.0};
    auto level = [&](int k, auto first, auto odd) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first)::value, ODD = decltype(odd)::value;
        const T *__restrict__ s = k == ns ? a.last : a.top - (size_t)(k - 1) * a.stride;
        const int hk = h + 2 * (ns - k), n = (w + 2 * (ns - k)) * hk;
        const float rh = 1.0f / float(hk);
        for (int i = threadIdx.x; i < n; i += NT) {
            double g[9], lam[9], mu[9];
            const Cell c = cell(k, i, hk, rh);
#pragma unroll
            for (int q = 0; q < 9; ++q)
                g[q] = double(load_pop<ST>(
                    reinterpret_cast<const T *>(reinterpret_cast<const char *>(s + q * L) +
                                                from(c, q, 1)),
                    a.inv_scale));
            double *m = mem + c.lx * 9 * H + c.ly;
#pragma unroll
            for (int q = 0; q < 9; ++q)
                if constexpr (FIRST) lam[q] = *mu_at(a.mu_in, q, from(c, q, -1));
                else lam[q] = ODD ? m[opposite(q) * H] : m[(q + 9 * cx(q)) * H + cy(q)];
            const double d = adj_cell<Traits<ST>::shifted>(g, lam, a.omega, mu);
            const int ox = c.lx - halo, oy = c.ly - halo;
            const bool own = ox >= 0 && ox < w && oy >= 0 && oy < h;
            if (own) sum.add(d);
            if (k == ns) {
                if (own)
#pragma unroll
                    for (int q = 0; q < 9; ++q) *mu_at(a.mu_out, q, c.c0 + c.r0) = mu[q];
            } else {
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if constexpr (FIRST || ODD) m[q * H] = mu[q];
                    else m[(q + 9 * cx(q)) * H + cy(q)] = mu[opposite(q)];
            }
        }
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    level(1, yes, no);
    for (int k = 2; k <= ns; ++k) {
        __syncthreads();
        if (k & 1) level(k, no, yes);
        else level(k, no, no);
    }
    sum = wave_sum(sum);
    if (first_lane) *mine = sum;
}

// One partial sum per workgroup, or of one workgroup the total.
__global__ void __launch_bounds__(256) k_adj_total(const Sum2 *in, size_t n, Sum2 *out,
                                                   double *total) {
    __shared__ Sum2 sh[4];
    Sum2 v{0.0, 0.0};
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        v.add(in[i]);
    v = block_sum<256>(v, sh);
    if (threadIdx.x == 0) {
        if (total) *total = v.value();
        else out[blockIdx.x] = v;
    }
}

// Gradient with respect to the initial macroscopic fields: f^0 = feq(rho0, u0),
// lambda^0_q(x) = mu^0_q(x + c_q).
__global__ void __launch_bounds__(256)
    k_adj_initial(const double *mu0, int nx, int ny, int ldd, const double *rho0, const double *ux0,
                  const double *uy0, double *grho, double *gux, double *guy) {
    const int y = blockIdx.x * blockDim.x + threadIdx.x, x = blockIdx.y;
    if (y >= ny) return;
    const size_t i = (size_t)x * ny + y;
    const double rho = rho0[i], ux = ux0[i], uy = uy0[i], u2 = ux * ux + uy * uy;
    double gr = 0, gx = 0, gy = 0;
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const double l = mu0[neighbour(x, y, q, nx, ny, ldd)] * wq(q);
        const double cu = cx(q) * ux + cy(q) * uy;
        gr += l * (1.0 + 3.0 * cu + 4.5 * cu * cu - 1.5 * u2);
        const double t = 3.0 + 9.0 * cu;
        gx += l * rho * (t * cx(q) - 3.0 * ux);
        gy += l * rho * (t * cy(q) - 3.0 * uy);
    }
    if (grho) grho[i] = gr;
    gux[i] = gx;
    guy[i] = gy;
}

__global__ void __launch_bounds__(256) k_adj_sum(const double *partials, int n, double *out) {
    __shared__ double sh[256];
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) a += partials[i];
    sh[threadIdx.x] = a;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0];
}

__global__ void __launch_bounds__(256) k_adj_zero(double *p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

}  // namespace plbm

using namespace plbm;

struct plbm_adjoint {
    int nx = 0, ny = 0, storage = 0, nsteps = 0, every = 0, ncheck = 0;
    plbm_lattice *lat = nullptr;   // forward buffers (ping-pong) + launch plumbing
    void *checkpoints = nullptr;   // ncheck buffers: f^0, f^K, f^2K, ...
    void *segment = nullptr;       // every buffers: the states of one segment after its first
    int held = -1;                 // the segment whose states it holds
    // The adjoint state: mu[0] of f^N, kept for further backward calls, and the two that a
    // reverse sweep alternates between (8-byte storages: the lattice's buffers, free by then).
    // Where FP32 storage has no memory for the third, the sweep overwrites mu[0].
    void *mu[3] = {nullptr, nullptr, nullptr};
    Sum2 *sums = nullptr;          // omega sensitivity, one per wavefront of a reverse pass
    size_t nsums = 0;              // the most wavefronts that one has
    size_t buf_bytes = 0, mu_bytes = 0;
    double omega = 0;
    bool forward_done = false;
    double *d_partials = nullptr;  // kAdjBlocks
    double *d_scalar = nullptr;    // 2
    const double *rho0 = nullptr, *ux0 = nullptr, *uy0 = nullptr;  // caller's device fields
    hipStream_t stream = nullptr;
};

namespace plbm {

static int adj_reduce_blocks(const plbm_adjoint *a) {
    const size_t n = (size_t)a->nx * a->ny;
    return (int)std::min<size_t>(kAdjBlocks, (n + 255) / 256);
}

static void *ckpt(plbm_adjoint *a, int k) {
    return static_cast<char *>(a->checkpoints) + (size_t)k * a->buf_bytes;
}
// f^{n0 + j} of segment k (n0 = k * every): its checkpoint or, once computed, from the buffer.
static void *state(plbm_adjoint *a, int k, int j) {
    return j == 0 ? ckpt(a, k) : static_cast<char *>(a->segment) + (size_t)(j - 1) * a->buf_bytes;
}

// The adjoint state is FP64 for every storage.
constexpr TileKind kAdjTiles{sizeof(double), PLBM_BGK};

// Depth of the object's passes.
static int adj_depth(const plbm_adjoint *a) {
    int shape, ns = 1;
    pick_tile(a->nx, a->ny, kAdjTiles, 1, kMaxStepsPerLaunch, &shape, &ns);
    return ns;
}
// f^{n0+1} .. f^{n0+len} of segment k from its checkpoint.
static int fill_segment(plbm_adjoint *a, int k, int len) {
    if (len < 1) return PLBM_OK;
    a->held = -1;
    int j = 0;
    for (int ns : pass_plan(len, adj_depth(a))) {
        PLBM_TRY(launch_tile_levels(a->lat, ns, state(a, k, j), state(a, k, j + 1)));
        j += ns;
    }
    a->held = k;
    return PLBM_OK;
}
// Tiles of a reverse pass of ns steps: shape, columns and rows of the grid of them.
static void adj_tiles(const plbm_adjoint *a, int ns, int *shape, int *nbx, int *nby) {
    int wx, wy;
    pick_tile(a->nx, a->ny, kAdjTiles, ns, ns, shape, &ns);
    tile_limits(*shape, ns, &wx, &wy);
    *nbx = (a->nx + wx - 1) / wx;
    *nby = (a->ny + wy - 1) / wy;
}
static size_t adj_waves(const plbm_adjoint *a, int ns) {
    int shape = 0, nbx, nby;
    adj_tiles(a, ns, &shape, &nbx, &nby);
    const int t = dispatch_tile_shape(shape, [](auto s) { return decltype(s)::T; });
    return (size_t)nbx * nby * (t / 64);
}

// One pass of ns reverse steps, states f^{top} (at `top`) down to the one at `last`.
static int launch_adj(plbm_adjoint *a, int ns, const void *top, const void *last, const void *in,
                      void *out) {
    const plbm_lattice *h = a->lat;
    int shape = 0, nbx, nby;
    adj_tiles(a, ns, &shape, &nbx, &nby);
    return dispatch_storage(a->storage, [&](auto S) {
        constexpr int SS = decltype(S)::value;
        if constexpr (SS == PLBM_F16S) {
            return PLBM_ERR_ARG;  // refused by plbm_adjoint_create
        } else {
            using T = typename Traits<SS>::T;
            AdjArgs<SS> g;
            g.top = static_cast<const T *>(top);
            g.last = static_cast<const T *>(last);
            g.stride = h->elems;
            g.cs = (size_t)9 * h->ldd;
            g.mu_in = static_cast<const double *>(in);
            g.mu_out = static_cast<double *>(out);
            g.partials = a->sums;
            g.nx = a->nx;
            g.ny = a->ny;
            g.ldd = h->ldd;
            g.omega = a->omega;
            g.inv_scale = float(1.0 / h->scale);
            // byte offsets within a state in 32 bits, columns multiplied in 24
            const bool near = h->elems * sizeof(double) < (1ull << 32) &&
                              g.cs * sizeof(T) < (1u << 24) && a->nx < (1 << 24);
            return dispatch_tile_shape(shape, [&](auto sh) {
                using SH = decltype(sh);
                auto go = [&](auto far_) {
                    hipLaunchKernelGGL((k_adj_tile<SS, SH, decltype(far_)::value>),
                                       dim3((unsigned)(nbx * nby)), dim3(SH::T), 0, a->stream, g,
                                       ns, nbx, nby);
                };
                if (near) go(std::false_type{});
                else go(std::true_type{});
                PLBM_HIP(hipGetLastError());
                return PLBM_OK;
            });
        }
    });
}

}  // namespace plbm

extern "C" {

int plbm_adjoint_create(int nx, int ny, int storage, int nsteps, int checkpoint_every,
                        plbm_adjoint **out) try {
    PLBM_REQUIRE(out, PLBM_ERR_ARG, "null output pointer");
    *out = nullptr;
    PLBM_REQUIRE(storage == PLBM_F64 || storage == PLBM_F64S || storage == PLBM_F32S,
                 PLBM_ERR_ARG, "adjoint storage must be F64, F64S or F32S");
    PLBM_REQUIRE(nsteps >= 1 && checkpoint_every >= 1, PLBM_ERR_ARG,
                 "nsteps and checkpoint_every must be >= 1");
    auto *a = new plbm_adjoint();
    a->nx = nx;
    a->ny = ny;
    a->storage = storage;
    a->nsteps = nsteps;
    a->every = std::min(checkpoint_every, nsteps);
    a->ncheck = (nsteps + a->every - 1) / a->every;  // checkpoints at 0, K, 2K, ... < N
    int st = plbm_create(nx, ny, 2, storage, &a->lat);
    if (st != PLBM_OK) {
        delete a;
        return st;
    }
    a->stream = a->lat->stream;
    a->buf_bytes = a->lat->elems * storage_bytes(storage);
    a->mu_bytes = a->lat->elems * sizeof(double);  // FP64 adjoint state for every storage
    for (int ns = 1; ns <= adj_depth(a); ++ns)
        a->nsums = std::max(a->nsums, adj_waves(a, ns));
    auto fail = [&](const char *m) {
        (void)hipGetLastError();
        set_error(m);
        plbm_adjoint_destroy(a);
        return PLBM_ERR_NOMEM;
    };
    if (hipMalloc(&a->checkpoints, a->ncheck * a->buf_bytes) != hipSuccess)
        return fail("hipMalloc of adjoint checkpoints failed");
    if (hipMalloc(&a->segment, a->every * a->buf_bytes) != hipSuccess)
        return fail("hipMalloc of the adjoint segment buffer failed");
    if (hipMalloc(&a->mu[0], a->mu_bytes) != hipSuccess ||
        hipMalloc(&a->sums, a->nsums * sizeof(Sum2)) != hipSuccess)
        return fail("hipMalloc of adjoint buffers failed");
    if (a->mu_bytes == a->buf_bytes) {
        a->mu[1] = a->lat->f[0];
        a->mu[2] = a->lat->f[1];
    } else if (hipMalloc(&a->mu[1], a->mu_bytes) != hipSuccess) {
        return fail("hipMalloc of adjoint buffers failed");
    }
    if (hipMalloc(&a->d_partials, kAdjBlocks * sizeof(double)) != hipSuccess ||
        hipMalloc(&a->d_scalar, 2 * sizeof(double)) != hipSuccess)
        return fail("hipMalloc of adjoint scalars failed");
    if (!a->mu[2] && hipMalloc(&a->mu[2], a->mu_bytes) != hipSuccess) {
        (void)hipGetLastError();
        a->mu[2] = nullptr;
    }
    *out = a;
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

int plbm_adjoint_destroy(plbm_adjoint *a) try {
    if (!a) return PLBM_OK;
    if (a->stream) (void)hipStreamSynchronize(a->stream);
    if (a->checkpoints) (void)hipFree(a->checkpoints);
    if (a->segment) (void)hipFree(a->segment);
    for (void *p : a->mu)
        if (p && p != a->lat->f[0] && p != a->lat->f[1]) (void)hipFree(p);
    if (a->sums) (void)hipFree(a->sums);
    if (a->d_partials) (void)hipFree(a->d_partials);
    if (a->d_scalar) (void)hipFree(a->d_scalar);
    if (a->lat) plbm_destroy(a->lat);
    delete a;
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

int plbm_adjoint_set_stream(plbm_adjoint *a, void *stream) try {
    PLBM_REQUIRE(a, PLBM_ERR_ARG, "null adjoint handle");
    PLBM_TRY(plbm_set_stream(a->lat, stream));
    a->stream = a->lat->stream;
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

int plbm_adjoint_forward_dev(plbm_adjoint *a, const double *rho0, const double *ux0,
                             const double *uy0, double omega, const double *uxt,
                             const double *uyt, double *loss) try {
    PLBM_REQUIRE(a && rho0 && ux0 && uy0 && uxt && uyt && loss, PLBM_ERR_ARG, "null argument");
    PLBM_REQUIRE(std::isfinite(omega), PLBM_ERR_ARG, "non-finite omega");
    plbm_lattice *h = a->lat;
    PLBM_TRY(plbm_set_params(h, omega, 0.25));
    a->forward_done = false;
    a->omega = omega;
    a->rho0 = rho0;
    a->ux0 = ux0;
    a->uy0 = uy0;
    PLBM_TRY(plbm_equilibrium_init_dev(h, 0, rho0, ux0, uy0));
    // each segment in tile passes from its checkpoint to the next; the last one's states, f^N
    // the last of them, stay in the segment buffer for the reverse sweep
    const int depth = adj_depth(a);
    const void *cur = h->f[0];
    PLBM_HIP(hipMemcpyAsync(ckpt(a, 0), cur, a->buf_bytes, hipMemcpyDeviceToDevice, a->stream));
    for (int k = 0; k + 1 < a->ncheck; ++k) {
        const std::vector<int> plan = pass_plan(a->every, depth);
        for (size_t p = 0; p < plan.size(); ++p) {
            void *to = p + 1 == plan.size() ? ckpt(a, k + 1) : cur == h->f[0] ? h->f[1] : h->f[0];
            PLBM_TRY(launch_tile(h, PLBM_BGK, plan[p], cur, to, nullptr, true));
            cur = to;
        }
    }
    const int len = a->nsteps - (a->ncheck - 1) * a->every;
    PLBM_TRY(fill_segment(a, a->ncheck - 1, len));
    cur = state(a, a->ncheck - 1, len);
    // loss and lambda^N
    const int nb = adj_reduce_blocks(a);
    PLBM_TRY(dispatch_storage(a->storage, [&](auto S) {
        constexpr int SS = decltype(S)::value;
        if constexpr (SS == PLBM_F16S) {
            set_error("adjoint: FP16 storage is not supported");
            return PLBM_ERR_ARG;
        } else {
            hipLaunchKernelGGL(k_adj_final<SS>, dim3(nb), dim3(256), 0, a->stream, cur, a->nx,
                               a->ny, h->ldd, float(1.0 / h->scale), uxt, uyt,
                               static_cast<double *>(a->mu[0]), a->d_partials);
            PLBM_HIP(hipGetLastError());
            return PLBM_OK;
        }
    }));
    hipLaunchKernelGGL(k_adj_sum, dim3(1), dim3(256), 0, a->stream, a->d_partials, nb, a->d_scalar);
    PLBM_HIP(hipGetLastError());
    PLBM_HIP(hipMemcpyAsync(loss, a->d_scalar, sizeof(double), hipMemcpyDeviceToHost, a->stream));
    PLBM_HIP(hipStreamSynchronize(a->stream));
    a->forward_done = true;
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

int plbm_adjoint_backward_dev(plbm_adjoint *a, double *grho0, double *gux0, double *guy0,
                              double *gomega) try {
    PLBM_REQUIRE(a && gux0 && guy0 && gomega, PLBM_ERR_ARG, "null argument");
    PLBM_REQUIRE(a->forward_done, PLBM_ERR_STATE, "run plbm_adjoint_forward_dev first");
    plbm_lattice *h = a->lat;
    hipLaunchKernelGGL(k_adj_zero, dim3((unsigned)((2 * a->nsums + 255) / 256)), dim3(256), 0,
                       a->stream, reinterpret_cast<double *>(a->sums), 2 * a->nsums);
    PLBM_HIP(hipGetLastError());
    const int depth = adj_depth(a);
    void *in = a->mu[0], *to = a->mu[1], *next = a->mu[2] ? a->mu[2] : a->mu[0];
    if (!a->mu[2]) a->forward_done = false;
    for (int k = a->ncheck - 1; k >= 0; --k) {
        const int n0 = k * a->every, n1 = std::min(a->nsteps, n0 + a->every);
        if (a->held != k) PLBM_TRY(fill_segment(a, k, n1 - n0 - 1));
        int top = n1 - 1 - n0;
        for (int ns : pass_plan(n1 - n0, depth)) {
            PLBM_TRY(launch_adj(a, ns, state(a, k, top), state(a, k, top - ns + 1), in, to));
            in = to;
            std::swap(to, next);
            top -= ns;
        }
    }
    // lambda^0 -> gradients of the initial fields
    hipLaunchKernelGGL(k_adj_initial, dim3((a->ny + 255) / 256, a->nx), dim3(256), 0, a->stream,
                       static_cast<const double *>(in), a->nx, a->ny, h->ldd, a->rho0,
                       a->ux0, a->uy0, grho0, gux0, guy0);
    PLBM_HIP(hipGetLastError());
    Sum2 *part = reinterpret_cast<Sum2 *>(a->d_partials);
    const int blocks = (int)std::min<size_t>(kAdjBlocks / 2, (a->nsums + 1023) / 1024);
    hipLaunchKernelGGL(k_adj_total, dim3(blocks), dim3(256), 0, a->stream, a->sums, a->nsums, part,
                       nullptr);
    PLBM_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_adj_total, dim3(1), dim3(256), 0, a->stream, part, (size_t)blocks,
                       nullptr, a->d_scalar + 1);
    PLBM_HIP(hipGetLastError());
    PLBM_HIP(hipMemcpyAsync(gomega, a->d_scalar + 1, sizeof(double), hipMemcpyDeviceToHost,
                            a->stream));
    PLBM_HIP(hipStreamSynchronize(a->stream));
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

}  // extern "C"
