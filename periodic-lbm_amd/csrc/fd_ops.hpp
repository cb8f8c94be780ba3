// fd_ops.hpp — the finite-volume / finite-difference streaming operators' kernels
// (src/fvm_bardow.F90:393-893) and their launchers, templated on the operator id, so that
// the operators can be instantiated in more than one translation unit (streaming_ops.hip:
// the default build's three operators; streaming_ops_fdm.hip: the -DFDM_* stencils;
// dugks.hip: DUGKS passes, which are the finite-volume update between half collisions).
#pragma once

#include <cmath>

#include <algorithm>
#include <utility>

#include "common.hpp"
#include "d2q9.hpp"
#include "multistep.hpp"
#include "stepper.hpp"
#include "tile.hpp"

namespace plbm {

// DUGKS steps as an operator of the pass kernels (dugks.hip): the window holds the
// half-collided state and the update is subtracted from the fully collided cell.  MODEL then
// says whether the two collisions differ (kDugksTwo) or have the same rate, as they have for
// dt = 1, so that one state serves both.
constexpr int kOpDugks = 100;
constexpr int kDugksOne = 0, kDugksTwo = 1;

// stream_fdm_bardow's stencil family: the 9-point first and second derivatives
// (src/fvm_bardow.F90:591-669).  PLBM_STREAM_FDM_BARDOW is the default build's central
// differences; the others are the variants the reference selects at compile time with
// -DFDM_WLS (weighted least squares, no weight), -DFDM_WLS_GAUSS_V1 / _V2 (Gaussian
// weights scaled to the farthest / closest node) and -DFDM_ISO (isotropic differences,
// Kumar 2004).  Each expression is grouped as Fortran evaluates it (left to right), with
// the reference's constants, so that FP64 results are bit-identical to those builds.
__host__ __device__ constexpr bool is_fdm_bardow(int op) {
    return op == PLBM_STREAM_FDM_BARDOW ||
           (op >= PLBM_STREAM_FDM_BARDOW_WLS && op <= PLBM_STREAM_FDM_BARDOW_ISO);
}

template <int OP, class R>
__device__ __forceinline__ void fdm_derivatives(R fc, R fe, R fn, R fw, R fs, R fne, R fnw,
                                                R fsw, R fse, R &dfx, R &dfy, R &dfxx, R &dfyy,
                                                R &dfxy) {
#pragma clang fp contract(off)
    const R two = R(2);
    if constexpr (OP == PLBM_STREAM_FDM_BARDOW) {
        const R p2 = R(0.5);
        dfx = p2 * (fe - fw);
        dfy = p2 * (fn - fs);
        dfxx = (fe - two * fc) + fw;
        dfyy = (fn - two * fc) + fs;
        dfxy = R(0.25) * (((fne - fse) - fnw) + fsw);
    } else if constexpr (OP == PLBM_STREAM_FDM_BARDOW_WLS) {
        const R one_sixth = R(1.0 / 6.0), one_third = R(1.0 / 3.0);
        dfx = one_sixth * (((fne - fnw) + (fe - fw)) + (fse - fsw));
        dfy = one_sixth * (((fne - fse) + (fn - fs)) + (fnw - fsw));
        dfxx = (one_third * ((fne - two * fn) + fnw) + one_third * ((fe - two * fc) + fw)) +
               one_third * ((fse - two * fs) + fsw);
        dfyy = (one_third * ((fne - two * fe) + fse) + one_third * ((fn - two * fc) + fs)) +
               one_third * ((fnw - two * fw) + fsw);
        dfxy = R(0.25) * (((fne - fnw) + fsw) - fse);
    } else if constexpr (OP == PLBM_STREAM_FDM_BARDOW_WLS_GAUSS_V1 ||
                         OP == PLBM_STREAM_FDM_BARDOW_WLS_GAUSS_V2) {
        constexpr bool v1 = OP == PLBM_STREAM_FDM_BARDOW_WLS_GAUSS_V1;
        const R p1s = v1 ? R(0.2880584423829145035434) : R(0.3934930210807994210853);
        const R p1d = v1 ? R(0.1059707788085427065949) : R(0.05325348945960039354075);
        const R p2c = v1 ? R(-1.152233769531658458263) : R(-1.573972084323197018207);
        const R p2d1 = v1 ? R(0.5761168847658292291314) : R(0.7869860421615988421706);
        const R p2d2 = v1 ? R(-0.4238831152341712149578) : R(-0.2130139578384016019186);
        const R p2d = v1 ? R(0.2119415576170855242122) : R(0.1065069789192007732037);
        dfx = (p1s * (fe - fw) + p1d * (fne - fnw)) + p1d * (fse - fsw);
        dfy = (p1s * (fn - fs) + p1d * (fne - fse)) + p1d * (fnw - fsw);
        const R corners = ((fne + fnw) + fsw) + fse;
        dfxx = ((p2c * fc + p2d1 * (fe + fw)) + p2d2 * (fn + fs)) + p2d * corners;
        dfyy = ((p2c * fc + p2d2 * (fe + fw)) + p2d1 * (fn + fs)) + p2d * corners;
        dfxy = R(0.25) * (((fne - fnw) + fsw) - fse);
    } else {
        static_assert(OP == PLBM_STREAM_FDM_BARDOW_ISO, "not an FDM Bardow stencil");
        const R p2 = R(0.5), one_sixth = R(1.0 / 6.0), two_thirds = R(2.0 / 3.0);
        const R five_sixths = R(10.0 / 12.0), one_twelfth = R(1.0 / 12.0);
        dfx = p2 * ((one_sixth * (fne - fnw) + two_thirds * (fe - fw)) + one_sixth * (fse - fsw));
        dfy = p2 * ((one_sixth * (fne - fse) + two_thirds * (fn - fs)) + one_sixth * (fnw - fsw));
        dfxx = (one_twelfth * ((fne - two * fn) + fnw) + five_sixths * ((fe - two * fc) + fw)) +
               one_twelfth * ((fse - two * fs) + fsw);
        dfyy = (one_twelfth * ((fne - two * fe) + fse) + five_sixths * ((fn - two * fc) + fs)) +
               one_twelfth * ((fnw - two * fw) + fsw);
        dfxy = R(0.25) * (((fne - fse) - fnw) + fsw);
    }
}

// Whether an operator's axis directions (cx or cy zero) carry terms that are zero times a
// difference of populations.
__host__ __device__ constexpr bool fd_zero_terms(int op) {
    return op == PLBM_STREAM_FVM_BARDOW || op == kOpDugks || is_fdm_bardow(op);
}

// One direction's update from its 3x3 neighbourhood (c = centre, e/n/w/s and corners); fp is
// the value it is subtracted from (fc but for DUGKS).  FINITE: the zero terms of the axis
// directions are left out.  For finite values they add +-0, so that the result is the same
// but for the sign of a zero; the pass kernels use it while everything a wavefront or tile
// has seen is finite and far from overflow.  It halves the finite-volume update (46 -> 13
// operations in four of eight directions) and drops those directions' neighbours.
template <int OP, class R, bool FINITE = false>
__device__ __forceinline__ R fd_update(int q, R fp, R fc, R fe, R fn, R fw, R fs, R fne, R fnw,
                                       R fsw, R fse, R dtr, R p2s) {
#pragma clang fp contract(off)
    if constexpr (fd_zero_terms(OP)) {
        const R cxq = dtr * R(cx(q)), cyq = dtr * R(cy(q));
        const bool along_x = FINITE && cy(q) == 0, along_y = FINITE && cx(q) == 0;
        if constexpr (!is_fdm_bardow(OP)) {
            const R p2 = R(0.5), p8 = R(0.125);
            R cfw = p2 * (fc + fw) - (p2 * cxq) * (fc - fw);
            R cfn = p2 * (fc + fn) - (p2 * cyq) * (fn - fc);
            R cfe = p2 * (fc + fe) - (p2 * cxq) * (fe - fc);
            R cfs = p2 * (fc + fs) - (p2 * cyq) * (fc - fs);
            if (along_x) return fp - cxq * (cfe - cfw);
            if (along_y) return fp - cyq * (cfn - cfs);
            cfw = cfw - (p8 * cyq) * (((fnw + fn) - fsw) - fs);
            cfn = cfn - (p8 * cxq) * (((fne + fe) - fnw) - fw);
            cfe = cfe - (p8 * cyq) * (((fne + fn) - fse) - fs);
            cfs = cfs - (p8 * cxq) * (((fse + fe) - fsw) - fw);
            return (fp - cxq * (cfe - cfw)) - cyq * (cfn - cfs);
        } else {
            const R cxxq = (R(0.5) * cxq) * cxq, cyyq = (R(0.5) * cyq) * cyq, cxyq = cxq * cyq;
            R dfx, dfy, dfxx, dfyy, dfxy;
            fdm_derivatives<OP, R>(fc, fe, fn, fw, fs, fne, fnw, fsw, fse, dfx, dfy, dfxx, dfyy,
                                   dfxy);
            if (along_x) return (fp - cxq * dfx) + cxxq * dfxx;
            if (along_y) return (fp - cyq * dfy) + cyyq * dfyy;
            return ((fp - cxq * dfx) - cyq * dfy) + ((cxxq * dfxx + cxyq * dfxy) + cyyq * dfyy);
        }
    } else {
        // fu at x + c_q (upstream of the pull), fd at x - c_q
        const int ux = cx(q), uy = cy(q);
        const R fu = ux > 0 ? (uy > 0 ? fne : (uy < 0 ? fse : fe))
                   : ux < 0 ? (uy > 0 ? fnw : (uy < 0 ? fsw : fw))
                            : (uy > 0 ? fn : fs);
        const R fd = ux > 0 ? (uy > 0 ? fsw : (uy < 0 ? fnw : fw))
                   : ux < 0 ? (uy > 0 ? fse : (uy < 0 ? fne : fe))
                            : (uy > 0 ? fs : fn);
        R du1, du2;
        if (q < 5) {
            du1 = R(0.5) * (fu - fd);
            du2 = (fu - R(2) * fc) + fd;
        } else {
            du1 = p2s * (fu - fd);
            du2 = R(0.5) * ((fu - R(2) * fc) + fd);
        }
        return fp + dtr * ((R(0.5) * dtr) * du2 - du1);
    }
}

// Each thread owns one row y and walks a strip of XS consecutive columns, keeping the
// 3x3 neighbourhood of every moving direction in registers, so that a step to the next
// column loads only that column's three values per direction.  MODEL < 0: streaming only,
// the rest population copied as stored.  MODEL >= 0: the streamed cell is collided before
// it is stored (perform_step's stream + collide pair in one pass; in FP64 storage the
// values are the unfused ones, since the unfused path stores the intermediate exactly).
template <int OP, int ST, int MODEL, int XS>
__global__ void __launch_bounds__(256)
    k_stream_fd(StepArgs a, double dt, double p2s) {
    using T = typename Traits<ST>::T;
    using R = typename Traits<ST>::R;
    const int y = blockIdx.x * 256 + threadIdx.x;
    const int x0 = blockIdx.y * XS;
    const int nx = a.nx, ny = a.ny;
    if (y >= ny) return;
    const T *__restrict__ s = static_cast<const T *>(a.src);
    T *__restrict__ d = static_cast<T *>(a.dst);
    const int ym = y == 0 ? ny - 1 : y - 1, yp = y == ny - 1 ? 0 : y + 1;
    const size_t L = (size_t)a.ldd, cs = a.cs;
    auto col = [&](int xx) {
        xx = xx < 0 ? xx + nx : (xx >= nx ? xx - nx : xx);
        return (size_t)xx * cs;
    };
    auto ld_ = [&](size_t c, int yy) { return load_pop<ST>(s + c + yy, a.inv_scale); };
    const R dtr = R(dt), p2r = R(p2s);
    R w[9][3][3];  // [q][column x-1, x, x+1][row y-1, y, y+1]; q = 0 unused
    {
        const size_t cm = col(x0 - 1), c0 = col(x0);
#pragma unroll
        for (int q = 1; q < 9; ++q) {
            const size_t o = (size_t)q * L;
            w[q][0][0] = ld_(cm + o, ym), w[q][0][1] = ld_(cm + o, y), w[q][0][2] = ld_(cm + o, yp);
            w[q][1][0] = ld_(c0 + o, ym), w[q][1][1] = ld_(c0 + o, y), w[q][1][2] = ld_(c0 + o, yp);
        }
    }
    for (int i = 0; i < XS; ++i) {
        const int x = x0 + i;
        if (x >= nx) break;
        const size_t c0 = (size_t)x * cs, cp = col(x + 1);
#pragma unroll
        for (int q = 1; q < 9; ++q) {
            const size_t o = (size_t)q * L;
            w[q][2][0] = ld_(cp + o, ym), w[q][2][1] = ld_(cp + o, y), w[q][2][2] = ld_(cp + o, yp);
        }
        R f[9];
#pragma unroll
        for (int q = 1; q < 9; ++q)
            f[q] = fd_update<OP, R>(q, w[q][1][1], w[q][1][1], w[q][2][1], w[q][1][2], w[q][0][1], w[q][1][0],
                                    w[q][2][2], w[q][0][2], w[q][0][0], w[q][2][0], dtr, p2r);
        if constexpr (MODEL < 0) {
            d[c0 + y] = s[c0 + y];
        } else {
            f[0] = ld_(c0, y);
            collide_cell<MODEL, ST>(f, a);
            store_pop<ST>(d + c0 + y, f[0], a.scale);
        }
#pragma unroll
        for (int q = 1; q < 9; ++q) {
            store_pop<ST>(d + c0 + (size_t)q * L + y, f[q], a.scale);
#pragma unroll
            for (int j = 0; j < 3; ++j) w[q][0][j] = w[q][1][j], w[q][1][j] = w[q][2][j];
        }
    }
}

// Scalars of the pass kernels beyond StepArgs.  A population sum of at least `big` in a cell
// (or a NaN) sends a wavefront or tile to the full update: below it every difference that the
// update multiplies, times dt and dt^2, stays finite.
struct FdScalars {
    double dt, p2s, big, om_half;
};
inline FdScalars fd_scalars(double dt, double om_half = 0.0) {
    const double t = 1.0 + std::fabs(dt);
    return {dt, 0.5 / std::sqrt(2.0) /* src/fvm_bardow.F90:712 */, 1e300 / (t * t), om_half};
}

// What the passes of an operator hold of a state f: the window value w (the state itself, or
// DUGKS's half-collided one) and, for kDugksTwo, the fully collided b.
template <int OP, int MODEL>
__device__ __forceinline__ void fd_enter(const double (&f)[9], double (&w)[9], double (&b)[9],
                                         const StepArgs &a, const FdScalars &s) {
#pragma unroll
    for (int q = 0; q < 9; ++q) w[q] = f[q];
    if constexpr (OP == kOpDugks) {
        collide_bgk_split_ref(w, s.om_half);
        if constexpr (MODEL == kDugksTwo) {
#pragma unroll
            for (int q = 0; q < 9; ++q) b[q] = f[q];
            collide_bgk_split_ref(b, a.omega);
        }
    }
}
template <int OP, int MODEL>
__device__ __forceinline__ void fd_collide(double (&f)[9], const StepArgs &a) {
    if constexpr (OP != kOpDugks) collide_cell<MODEL, PLBM_F64>(f, a);
}
// Whether every population of the cell is finite and far from overflow.
__device__ __forceinline__ bool fd_tame(const double (&f)[9], double big) {
    double t = fabs(f[0]);
#pragma unroll
    for (int q = 1; q < 9; ++q) t += fabs(f[q]);
    return t < big;
}

// NS steps of (streaming operator OP, collision MODEL) per sweep over device memory, FP64
// storage (temporal blocking as the lattice Boltzmann pass kernel): a wavefront owns 64
// consecutive rows (56 with output, NS halo rows on each side) and walks one of m segments of
// columns, keeping for every level k < NS the last three columns of its own row in registers;
// y-neighbours come from the adjacent lanes (DPP).  The columns are staged in LDS two ahead of
// the walk.  When level k receives a column, level k+1 gets the column before it: the
// operator's 3x3 stencil per direction, then the collision, exactly as k_stream_fd<OP, F64,
// MODEL> computes them (DUGKS: as k_dugks_collide and k_dugks_flux do).
// Bound by instruction issue at two wavefronts per SIMD (more do not fit its LDS): leaving out
// the zero terms took the finite-volume pass from 254 to 226 registers and, at 8192^2 with
// BGK, from 1.61 to 1.20 ms per step in passes of 3 and 1.16 in passes of 4, which now fit;
// stream_fdm_bardow 1.20 -> 0.89, stream_fdm_sofonea (no zero terms) 0.75 -> 0.67.
// `lag`: the state one step before the pass's last, or for DUGKS its half-collided form, which
// is what the other slot holds after a step.
template <int OP, int MODEL, int NS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
    k_fd_walk(StepArgs a, FdScalars sc, int waves_y, int m) {
    constexpr int VR = 56;
    static_assert(VR + 2 * NS <= 64, "halo rows do not fit in a wavefront");
    constexpr bool dugks = OP == kOpDugks, two = dugks && MODEL == kDugksTwo;
    const int lane = threadIdx.x & 63;
    const int gw = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (gw >= waves_y * m) return;  // the whole wavefront
    const int nx = a.nx, ny = a.ny;
    const int wy = gw % waves_y, seg = gw / waves_y;
    const int r = VR * wy - NS + lane;
    int y = r % ny;
    if (y < 0) y += ny;
    const bool out = lane >= NS && lane < VR + NS && r < ny;
    const int x0 = part_start(nx, m, seg), ncols = part_start(nx, m, seg + 1) - x0;
    const size_t L = (size_t)a.ldd, cs = a.cs;
    const double *__restrict__ s = static_cast<const double *>(a.src);
    double *__restrict__ d = static_cast<double *>(a.dst);
    double *__restrict__ lag = static_cast<double *>(a.lag);  // wave-uniform
    auto column = [&](int c) {
        c %= nx;
        if (c < 0) c += nx;
        return (size_t)c * cs;
    };
    double W[NS][3][9];          // [level][newest column, -1, -2][q], own row
    double F[two ? NS : 1][9];   // fully collided state of each level's newest column
#pragma unroll
    for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int q = 0; q < 9; ++q) W[k][j][q] = 0.0;
#pragma unroll
    for (int k = 0; k < (two ? NS : 1); ++k)
#pragma unroll
        for (int q = 0; q < 9; ++q) F[k][q] = 0.0;
    // set, wave-uniform, by the first column of any level that is not tame: every stencil that
    // reads it or a later column then takes the full update
    bool full = false;
    auto check = [&](const double(&f)[9]) __attribute__((always_inline)) {
        if constexpr (fd_zero_terms(OP)) full |= __ballot(!fd_tame(f, sc.big)) != 0;
    };
    const int iters = ncols + 2 * NS;
    // the next columns are staged in LDS ahead of the walk (as in the LBM pass kernel),
    // so their latency overlaps the operator and collisions of the current column
    ColumnStage st{};
    st.init(stage_buffers(), s, L, ny, VR * wy - NS, lane);
#pragma unroll
    for (int j = 0; j < kStageAhead; ++j)
        if (j < iters) st.fetch(s, column(x0 - NS + j), L, j % kStageBufs);
    for (int i = 0; i < iters; ++i) {
        double f[9];
        // (DUGKS stores both outputs in the same iterations; counting one of them makes the
        // wait the stronger)
        st.wait(i, iters, 2 * NS, !dugks && a.lag != nullptr);
        {
            const double *slot = st.column(i);
#pragma unroll
            for (int q = 0; q < 9; ++q) f[q] = slot[q * 64 + lane];
        }
        if (i + kStageAhead < iters)
            st.fetch(s, column(x0 - NS + i + kStageAhead), L, (i + kStageAhead) % kStageBufs);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (i < 2 * k) break;  // level k has no column yet
            double w[9], b[9], bprev[9];
            fd_enter<OP, MODEL>(f, w, b, a, sc);
            check(w);
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                W[k][2][q] = W[k][1][q];
                W[k][1][q] = W[k][0][q];
                W[k][0][q] = w[q];
                if constexpr (two) {
                    bprev[q] = F[k][q];
                    F[k][q] = b[q];
                } else {
                    bprev[q] = W[k][1][q];
                }
            }
            if (i < 2 * k + 2) break;  // level k+1 needs three columns of level k
            f[0] = bprev[0];
            auto stencil = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
                for (int q = 1; q < 9; ++q) {
                    const double fc = W[k][1][q], fe = W[k][0][q], fw = W[k][2][q];
                    f[q] = fd_update<OP, double, decltype(finite)::value>(
                        q, bprev[q], fc, fe, row_plus(fc), fw, row_minus(fc), row_plus(fe),
                        row_plus(fw), row_minus(fw), row_minus(fe), sc.dt, sc.p2s);
                }
            };
            if (full) stencil(std::false_type{});
            else stencil(std::bool_constant<fd_zero_terms(OP)>{});
            fd_collide<OP, MODEL>(f, a);
            if (k + 1 == NS && out) {
                const size_t co = (size_t)(x0 - 2 * NS + i) * cs + y;
#pragma unroll
                for (int q = 0; q < 9; ++q) __builtin_nontemporal_store(f[q], d + co + q * L);
                if (dugks && lag != nullptr)
#pragma unroll
                    for (int q = 0; q < 9; ++q)
                        __builtin_nontemporal_store(W[k][1][q], lag + co + q * L);
            } else if (!dugks && k + 2 == NS && lag != nullptr && i >= 2 * NS - 1 &&
                       i < 2 * NS - 1 + ncols && out) {
                // level NS-1 (the state one step before the pass's last) of column
                // x0 + i - (2 NS - 1)
                const size_t co = (size_t)(x0 - 2 * NS + 1 + i) * cs + y;
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    __builtin_nontemporal_store(f[q], lag + co + q * L);
            }
        }
    }
}

// The same ns steps of one tile held in LDS (one thread per cell and round, as tile.hpp's;
// the stencils read the neighbours of every direction, so that a level's results wait in
// registers until all of its reads are done).  Bound by instruction issue (75% of the slots)
// with the LDS reads, 48 per cell without the zero terms' and 72 with, half hidden beside it.
// It needs fewer cells than the walk to fill the chip; us per step with BGK, single steps /
// walk / tiles: 128^2 FVM 5.2 / - / 2.5, FDM 4.6 / - / 2.3, 400^2 FVM 15.8 / 13.4 / 5.3, FDM
// 15.2 / 11.6 / 4.7, 1000^2 FVM 55 / 24.5 / 22.8, FDM 55 / 20.2 / 19.6, Sofonea 32 / 15.7 /
// 15.2; 2048^2 FVM 152 / 77.5 / 82.4, FDM 153 / 61 / 73, Sofonea 127 / 45 / 58.  Two to four
// columns per thread, to read shared neighbours once, took more than 256 registers (40-90%
// slower); rows padded to 32 lanes remove the bank conflicts (a third of the LDS time) for 8%
// more instructions, and measured the same.
template <int XW_, int H_, int T_>
struct FdShape {
    static constexpr int XW = XW_, H = H_, T = T_;
};
using FdTileS = FdShape<24, 24, 512>;
using FdTileM = FdShape<34, 33, 512>;
template <int OP, int MODEL, class SHAPE>
__global__ void __launch_bounds__(SHAPE::T) __attribute__((amdgpu_waves_per_eu(4)))
    k_fd_tile(StepArgs a, FdScalars sc, int ns, int nbx, int nby) {
    constexpr int XW = SHAPE::XW, H = SHAPE::H, NT = SHAPE::T;
    constexpr int C = ((XW - 2) * (H - 2) + NT - 1) / NT;  // cells of a thread at level 1
    constexpr bool dugks = OP == kOpDugks, two = dugks && MODEL == kDugksTwo;
    __shared__ double mem[XW * 9 * H];                 // window values, (lx, q, ly)
    __shared__ double memb[two ? XW * 9 * H : 1];      // fully collided state
    __shared__ int full_sh;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int by = bid % nby, bx = bid / nby;
    const int x0 = part_start(a.nx, nbx, bx), w = part_start(a.nx, nbx, bx + 1) - x0;
    const int y0 = part_start(a.ny, nby, by), h = part_start(a.ny, nby, by + 1) - y0;
    const double *__restrict__ s = static_cast<const double *>(a.src);
    double *__restrict__ d = static_cast<double *>(a.dst);
    double *__restrict__ lag = static_cast<double *>(a.lag);
    const size_t L = (size_t)a.ldd;
    if (threadIdx.x == 0) full_sh = 0;
    bool wild = false;  // this thread has met a cell that is not tame
    auto check = [&](const double(&f)[9]) __attribute__((always_inline)) {
        if constexpr (fd_zero_terms(OP)) wild |= !fd_tame(f, sc.big);
    };
    {
        const int h0 = h + 2 * ns, n = (w + 2 * ns) * h0;
        const float rh = 1.0f / float(h0);
        for (int i = threadIdx.x; i < n; i += NT) {
            const int lx = int((float(i) + 0.5f) * rh), ly = i - lx * h0;
            const int x = wrap_index(x0 - ns + lx, a.nx), y = wrap_index(y0 - ns + ly, a.ny);
            const double *p = s + (size_t)x * a.cs + y;
            double f[9], v[9], b[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) f[q] = p[q * L];
            fd_enter<OP, MODEL>(f, v, b, a, sc);
            check(v);
            const int o = lx * 9 * H + ly;
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                mem[o + q * H] = v[q];
                if constexpr (two) memb[o + q * H] = b[q];
            }
        }
    }
    __syncthreads();  // full_sh is cleared
    for (int k = 1; k <= ns; ++k) {
        if (wild) full_sh = 1;
        __syncthreads();
        const bool full = full_sh != 0;
        const int hk = h + 2 * (ns - k), n = (w + 2 * (ns - k)) * hk;
        const float rh = 1.0f / float(hk);
        double f[C][9];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = threadIdx.x + c * NT;
            if (i < n) {
                const int ix = int((float(i) + 0.5f) * rh);
                const int lx = ix + k, ly = i - ix * hk + k;
                const double *m = mem + lx * 9 * H + ly;
                const double *mb = two ? memb + lx * 9 * H + ly : m;
                f[c][0] = mb[0];
                auto stencil = [&](auto finite) __attribute__((always_inline)) {
#pragma unroll
                    for (int q = 1; q < 9; ++q) {
                        const double *p = m + q * H;
                        f[c][q] = fd_update<OP, double, decltype(finite)::value>(
                            q, mb[q * H], p[0], p[9 * H], p[1], p[-9 * H], p[-1], p[9 * H + 1],
                            p[-9 * H + 1], p[-9 * H - 1], p[9 * H - 1], sc.dt, sc.p2s);
                    }
                };
                if (full) stencil(std::false_type{});
                else stencil(std::bool_constant<fd_zero_terms(OP)>{});
                fd_collide<OP, MODEL>(f[c], a);
                const int ox = lx - ns, oy = ly - ns;
                if (k >= ns - 1 && ox >= 0 && ox < w && oy >= 0 && oy < h) {
                    const size_t o = (size_t)(x0 + ox) * a.cs + (y0 + oy);
                    double *to = k == ns ? d : dugks ? nullptr : lag;
                    if (to != nullptr)
#pragma unroll
                        for (int q = 0; q < 9; ++q) to[o + q * L] = f[c][q];
                    if (dugks && k == ns && lag != nullptr)
#pragma unroll
                        for (int q = 0; q < 9; ++q) lag[o + q * L] = m[q * H];
                }
            }
        }
        if (k == ns) break;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = threadIdx.x + c * NT;
            if (i < n) {
                const int ix = int((float(i) + 0.5f) * rh);
                const int o = (ix + k) * 9 * H + (i - ix * hk + k);
                double v[9], b[9];
                fd_enter<OP, MODEL>(f[c], v, b, a, sc);
                check(v);
#pragma unroll
                for (int q = 0; q < 9; ++q) {
                    mem[o + q * H] = v[q];
                    if constexpr (two) memb[o + q * H] = b[q];
                }
            }
        }
    }
}

inline StepArgs fd_args(const plbm_lattice *h, const void *src, void *dst) {
    StepArgs a{};
    a.src = src;
    a.dst = dst;
    a.nx = h->nx;
    a.ny = h->ny;
    a.ldd = h->ldd;
    a.nby = (h->ny + 255) / 256;
    a.cs = (size_t)9 * h->ldd;
    a.omega = h->omega;
    a.lambda_odd = h->lambda_odd;
    a.omega_f = float(h->omega);
    a.lambda_odd_f = float(h->lambda_odd);
    a.scale = float(h->scale);
    a.inv_scale = float(1.0 / h->scale);
    return a;
}

// One launch of operator OP (+ collision `model`; model < 0: streaming only), src -> dst.
template <int OP>
int launch_fd_op(plbm_lattice *h, int model, const void *src, void *dst, double dt) {
    const double p2s = 0.5 / std::sqrt(2.0);  // src/fvm_bardow.F90:712
    const StepArgs a = fd_args(h, src, dst);
    const int xs = strip_columns(h->nx, h->ny);
    const dim3 grid((unsigned)a.nby, (unsigned)((h->nx + xs - 1) / xs));
    return dispatch_storage(h->storage, [&](auto S) {
        constexpr int SS = decltype(S)::value;
        auto go = [&](auto M) {
            constexpr int MM = decltype(M)::value;
            if (xs == 32)
                hipLaunchKernelGGL((k_stream_fd<OP, SS, MM, 32>), grid, dim3(256), 0, h->stream, a,
                                   dt, p2s);
            else if (xs == 8)
                hipLaunchKernelGGL((k_stream_fd<OP, SS, MM, 8>), grid, dim3(256), 0, h->stream, a,
                                   dt, p2s);
            else
                hipLaunchKernelGGL((k_stream_fd<OP, SS, MM, 1>), grid, dim3(256), 0, h->stream, a,
                                   dt, p2s);
            return 0;
        };
        switch (model) {
        case PLBM_BGK: go(std::integral_constant<int, PLBM_BGK>{}); break;
        case PLBM_TRT: go(std::integral_constant<int, PLBM_TRT>{}); break;
        case PLBM_RR: go(std::integral_constant<int, PLBM_RR>{}); break;
        case PLBM_BGK_SPLIT: go(std::integral_constant<int, PLBM_BGK_SPLIT>{}); break;
        default: go(std::integral_constant<int, -1>{});
        }
        PLBM_HIP(hipGetLastError());
        return PLBM_OK;
    });
}

// Grids of up to this many cells run the passes of the streaming operators in tiles.
constexpr long long kFdTileCells = 1000000;
constexpr int kFdWalkSteps = 4;  // deepest walk
constexpr int kFdTileSteps = 6;  // deepest tile chosen

// Shape (0 S, 1 M) and depth in [ns_min, ns_max] of the cheapest tile passes.  A CU with n
// tiles takes n + 0.3 (M) or n + 0.6 (S) times a tile's steps, as a single tile per CU cannot
// hide its latency, at 4.3 ns per cell (FVM + BGK); a launch costs 700 steps of a cell.
inline void pick_fd_tile(int nx, int ny, int ns_min, int ns_max, bool small_only, int *shape,
                         int *ns) {
    double best = 1e300;
    for (int n = ns_min; n <= ns_max; ++n)
        for (int s = 0; s < (small_only ? 1 : 2); ++s) {
            const int wx = (s ? FdTileM::XW : FdTileS::XW) - 2 * n;
            const int wy = (s ? FdTileM::H : FdTileS::H) - 2 * n;
            const long long nbx = (nx + wx - 1) / wx, nby = (ny + wy - 1) / wy;
            const double w = double((nx + nbx - 1) / nbx), h = double((ny + nby - 1) / nby);
            double c = 0.15 * ((w + 2 * n) * (h + 2 * n) + w * h);
            for (int k = 0; k < n; ++k) c += (w + 2 * k) * (h + 2 * k);
            const double per_cu = double((nbx * nby + kComputeUnits - 1) / kComputeUnits);
            const double t = (700 + c * (per_cu + (s ? 0.3 : 0.6))) / n;
            if (t < best) {
                best = t;
                *shape = s;
                *ns = n;
            }
        }
}

// One pass of ns steps of (OP, MODEL), FP64 storage; with a.lag set it also stores the state
// one step before its last (DUGKS: that state's half-collided form) there.
template <int OP, int MODEL>
int launch_fd_tile(plbm_lattice *h, int ns, const StepArgs &a, const FdScalars &sc) {
    constexpr bool small_only = OP == kOpDugks && MODEL == kDugksTwo;  // two states in LDS
    int shape = 0;
    pick_fd_tile(h->nx, h->ny, ns, ns, small_only, &shape, &ns);
    auto go = [&](auto sh) {
        using SH = decltype(sh);
        const int wx = SH::XW - 2 * ns, wy = SH::H - 2 * ns;
        const int nbx = (h->nx + wx - 1) / wx, nby = (h->ny + wy - 1) / wy;
        hipLaunchKernelGGL((k_fd_tile<OP, MODEL, SH>), dim3((unsigned)(nbx * nby)), dim3(SH::T),
                           0, h->stream, a, sc, ns, nbx, nby);
    };
    if constexpr (!small_only) {
        if (shape == 1) {
            go(FdTileM{});
            PLBM_HIP(hipGetLastError());
            return PLBM_OK;
        }
    }
    go(FdTileS{});
    PLBM_HIP(hipGetLastError());
    return PLBM_OK;
}
template <int OP, int MODEL, int NS>
int launch_fd_walk(plbm_lattice *h, const StepArgs &a, const FdScalars &sc) {
    const int bands = (h->ny + 55) / 56;
    const int m = pass_segments(h->nx, bands, NS, 8, 2, 1.0);
    const dim3 grid((unsigned)(((long long)bands * m + 3) / 4));
    hipLaunchKernelGGL((k_fd_walk<OP, MODEL, NS>), grid, dim3(256), 0, h->stream, a, sc, bands,
                       m);
    PLBM_HIP(hipGetLastError());
    return PLBM_OK;
}

// Long grids of few columns, whose tiles are mostly halo, keep single steps: us per step, FVM + BGK,
// runs of 4 / 40 steps, single steps and tiles: 1 x 25000 8.0 / 5.4, 9.6 / 6.9, 2 x 60000 11.8 /
// 9.3, 17.5 / 14.6, 4 x 60000 18.7 / 16.0, 19.4 / 16.4; but 3 x 25000 11.3 / 8.7, 9.9 / 7.1, 6 x
// 60000 26 / 23, 19.7 / 16.9.
inline bool fd_slender(const plbm_lattice *h) {
    return h->nx <= 4 && h->ny > 8192 * (h->nx + 1);
}
inline bool fd_tile_grid(const plbm_lattice *h) {
    return (long long)h->nx * h->ny <= kFdTileCells && !fd_slender(h);
}

// One pass of ns steps (2 .. kFdTileSteps in tiles, 2 .. kFdWalkSteps in walks) of operator
// OP and `model`.
template <int OP>
int launch_fd_multi_op(plbm_lattice *h, int model, int ns, const void *src, void *dst,
                       double dt, void *lag) {
    StepArgs a = fd_args(h, src, dst);
    a.lag = lag;
    const FdScalars sc = fd_scalars(dt);
    return dispatch_model(model, [&](auto M) {
        constexpr int MM = decltype(M)::value;
        if (fd_tile_grid(h)) return launch_fd_tile<OP, MM>(h, ns, a, sc);
        if (ns == 2) return launch_fd_walk<OP, MM, 2>(h, a, sc);
        if (ns == 3) return launch_fd_walk<OP, MM, 3>(h, a, sc);
        return launch_fd_walk<OP, MM, 4>(h, a, sc);
    });
}

// The -DFDM_* stencils (streaming_ops_fdm.hip): op in PLBM_STREAM_FDM_BARDOW_WLS ..
// PLBM_STREAM_FDM_BARDOW_ISO.
int launch_fd_variant(plbm_lattice *h, int op, int model, const void *src, void *dst, double dt);
int launch_fd_multi_variant(plbm_lattice *h, int op, int model, int ns, const void *src,
                            void *dst, double dt, void *lag);

}  // namespace plbm
