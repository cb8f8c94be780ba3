// streaming_ops.hip — the reference's finite-volume / finite-difference streaming
// operators on the device, for the grid%streaming slot (src/fvm_bardow.F90:393-893):
//   PLBM_STREAM_FVM_BARDOW   stream_fvm_bardow  (bilinear face fluxes, :410-509)
//   PLBM_STREAM_FDM_BARDOW   stream_fdm_bardow  (central-difference Lax-Wendroff, default
//                                                stencil without FDM_* options, :526-685)
//   PLBM_STREAM_FDM_SOFONEA  stream_fdm_sofonea (1-D Lax-Wendroff along c_q, :702-889)
//   PLBM_STREAM_FDM_BARDOW_WLS .. _ISO  stream_fdm_bardow built with -DFDM_WLS,
//                            -DFDM_WLS_GAUSS_V1, -DFDM_WLS_GAUSS_V2, -DFDM_ISO (:591-669;
//                            instantiated in streaming_ops_fdm.hip)
// Each is a 9-point (3-point for Sofonea) stencil on one q-segment of the column-
// interleaved layout; the rest population is copied.  plbm_step_op fuses the operator with
// the collision that perform_step applies next (one pass, 144 bytes per cell in FP64).
// The operators are linear and leave constants unchanged, so they act on shifted and
// scaled storage directly.  FP64 expression trees follow the reference with FMA
// contraction off, which makes them bit-identical to it.  The reference loops x over ny
// and y over nx (square grids); here x runs over nx and y over ny.
#include <algorithm>
#include <string>
#include <vector>

#include "fd_ops.hpp"

using namespace plbm;

namespace {

// model < 0: streaming only
int launch_fd(plbm_lattice *h, int op, int model, const void *src, void *dst, double dt) {
    switch (op) {
    case PLBM_STREAM_FVM_BARDOW:
        return launch_fd_op<PLBM_STREAM_FVM_BARDOW>(h, model, src, dst, dt);
    case PLBM_STREAM_FDM_BARDOW:
        return launch_fd_op<PLBM_STREAM_FDM_BARDOW>(h, model, src, dst, dt);
    case PLBM_STREAM_FDM_SOFONEA:
        return launch_fd_op<PLBM_STREAM_FDM_SOFONEA>(h, model, src, dst, dt);
    default:
        return launch_fd_variant(h, op, model, src, dst, dt);
    }
}

int launch_fd_multi(plbm_lattice *h, int op, int model, int ns, const void *src, void *dst,
                    double dt, void *lag = nullptr) {
    switch (op) {
    case PLBM_STREAM_FVM_BARDOW:
        return launch_fd_multi_op<PLBM_STREAM_FVM_BARDOW>(h, model, ns, src, dst, dt, lag);
    case PLBM_STREAM_FDM_BARDOW:
        return launch_fd_multi_op<PLBM_STREAM_FDM_BARDOW>(h, model, ns, src, dst, dt, lag);
    case PLBM_STREAM_FDM_SOFONEA:
        return launch_fd_multi_op<PLBM_STREAM_FDM_SOFONEA>(h, model, ns, src, dst, dt, lag);
    default:
        return launch_fd_multi_variant(h, op, model, ns, src, dst, dt, lag);
    }
}

int check_op_args(plbm_lattice *h, int op, int src, int dst, double dt) {
    PLBM_REQUIRE(h, PLBM_ERR_ARG, "null lattice handle");
    PLBM_REQUIRE(src >= 0 && src < h->nf && dst >= 0 && dst < h->nf && src != dst, PLBM_ERR_ARG,
                 "need distinct valid src and dst buffers");
    PLBM_REQUIRE(std::isfinite(dt), PLBM_ERR_ARG, "non-finite dt");
    PLBM_REQUIRE(op >= PLBM_STREAM_EXACT && op <= PLBM_STREAM_FDM_BARDOW_ISO, PLBM_ERR_ARG,
                 "unknown streaming operator " + std::to_string(op));
    note_capture(h);
    return PLBM_OK;
}

}  // namespace

extern "C" int plbm_stream_op(plbm_lattice *h, int op, int src, int dst, double dt) try {
    PLBM_TRY(check_op_args(h, op, src, dst, dt));
    if (op == PLBM_STREAM_EXACT) return plbm_stream(h, src, dst);
    return launch_fd(h, op, -1, h->f[src], h->f[dst], dt);
} catch (...) {
    return plbm::host_exception();
}

extern "C" int plbm_step_op(plbm_lattice *h, int op, int model, int src, int dst, double dt) try {
    PLBM_TRY(check_op_args(h, op, src, dst, dt));
    PLBM_REQUIRE(model >= PLBM_BGK && model <= PLBM_BGK_SPLIT, PLBM_ERR_ARG,
                 "unknown collision model " + std::to_string(model));
    PLBM_REQUIRE(h->params_set, PLBM_ERR_STATE, "plbm_set_params has not been called");
    if (op == PLBM_STREAM_EXACT) return plbm_step(h, model, src, dst);
    return launch_fd(h, op, model, h->f[src], h->f[dst], dt);
} catch (...) {
    return plbm::host_exception();
}

// Grids on which a captured run (plbm_lattice::captured) takes single steps, whose slots do not
// move; on others it takes passes of 3.  A graph is then replayed from the slots it was captured
// with, whatever the automatic depth of other runs is.
static bool fd_few_walks(const plbm_lattice *h) {
    return (long)((h->ny + 55) / 56) * ((h->nx + kMultiXS - 1) / kMultiXS) < 2048;
}

// Steps per pass of plbm_run_op when the caller has not chosen (FP64 storage; else single
// steps): walks of 4, the most that fit (8192^2, ms per step with BGK in passes of 2 / 3 / 4:
// FVM 1.22 / 1.20 / 1.16, FDM 1.04 / 0.96 / 0.89, Sofonea 0.95 / 0.74 / 0.67), or tiles of the
// cheapest depth on small grids.
static int fd_steps_per_pass(const plbm_lattice *h) {
    if (h->fd_ns > 0) return h->fd_ns;
    if (h->storage != PLBM_F64) return 1;
    if (fd_slender(h) && fd_few_walks(h)) return 1;
    if (!fd_tile_grid(h)) return kFdWalkSteps;
    int shape, ns = 2;
    pick_fd_tile(h->nx, h->ny, 2, kFdTileSteps, false, &shape, &ns);
    return ns;
}

extern "C" int plbm_set_op_steps_per_pass(plbm_lattice *h, int steps) try {
    PLBM_REQUIRE(h, PLBM_ERR_ARG, "null lattice handle");
    PLBM_REQUIRE(steps >= 0 && steps <= 3, PLBM_ERR_ARG, "steps per pass must be 0..3");
    PLBM_REQUIRE(steps <= 1 || h->storage == PLBM_F64, PLBM_ERR_STATE,
                 "passes of the streaming operators need FP64 (PLBM_F64) storage");
    h->fd_ns = steps;
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

extern "C" int plbm_get_op_steps_per_pass(const plbm_lattice *h, int op, int model,
                                          int *steps) try {
    PLBM_REQUIRE(h && steps, PLBM_ERR_ARG, "null argument");
    (void)op;
    (void)model;
    *steps = std::min(fd_steps_per_pass(h), 3);
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}

extern "C" int plbm_run_op(plbm_lattice *h, int op, int model, int nsteps, int *iold,
                           int *inew, double dt) try {
    PLBM_REQUIRE(h && iold && inew, PLBM_ERR_ARG, "null argument");
    PLBM_REQUIRE(nsteps >= 0, PLBM_ERR_ARG, "nsteps must be >= 0");
    PLBM_TRY(check_op_args(h, op, *iold, *inew, dt));
    PLBM_REQUIRE(model >= PLBM_BGK && model <= PLBM_BGK_SPLIT, PLBM_ERR_ARG,
                 "unknown collision model " + std::to_string(model));
    PLBM_REQUIRE(h->params_set, PLBM_ERR_STATE, "plbm_set_params has not been called");
    if (op == PLBM_STREAM_EXACT) return plbm_run(h, model, nsteps, iold, inew);
    int ns = fd_steps_per_pass(h);
    const bool fixed = h->fd_ns == 0 && h->captured;
    if (fixed && ns > 1) ns = fd_few_walks(h) ? 1 : 3;
    const bool even = h->fd_ns == 0 && !fixed && fd_tile_grid(h);
    if (ns <= 1 || nsteps < 2) {
        for (int s = 0; s < nsteps; ++s) {
            PLBM_TRY(launch_fd(h, op, model, h->f[*iold], h->f[*inew], dt));
            std::swap(*iold, *inew);
        }
        return PLBM_OK;
    }
    // passes of up to ns steps; the last, as deep as a pass goes, also stores the state one
    // step before the latest into the third buffer, which becomes the other slot's storage
    // (as after perform_step).  Without a third buffer the last step is a single fused step
    // instead.
    const int a0 = *iold, b0 = *inew;
    void *latest = h->f[a0], *other = h->f[b0];
    void *aux = pass_aux(h);
    const std::vector<int> plan = !aux   ? pass_plan(nsteps - 1, ns)
                                  : even ? pass_plan(nsteps, ns)
                                         : lag_pass_plan(nsteps, ns);
    for (size_t p = 0; p + 1 < plan.size(); ++p) {
        if (plan[p] == 1) PLBM_TRY(launch_fd(h, op, model, latest, other, dt));
        else PLBM_TRY(launch_fd_multi(h, op, model, plan[p], latest, other, dt));
        std::swap(latest, other);
    }
    if (aux) {
        PLBM_TRY(launch_fd_multi(h, op, model, plan.back(), latest, other, dt, aux));
        finish_run(h, a0, b0, nsteps, other, aux, latest, iold, inew);
        return PLBM_OK;
    }
    if (plan.back() == 1) PLBM_TRY(launch_fd(h, op, model, latest, other, dt));
    else PLBM_TRY(launch_fd_multi(h, op, model, plan.back(), latest, other, dt));
    std::swap(latest, other);
    PLBM_TRY(launch_fd(h, op, model, latest, other, dt));
    finish_run(h, a0, b0, nsteps, other, latest, nullptr, iold, inew);
    return PLBM_OK;
} catch (...) {
    return plbm::host_exception();
}
