"""The column walk of plbm_run's passes, which small grids take only when the caller sets their
column segments, and its automatic split on ragged grids just beyond those that run in tiles:
every model, depth and storage, the lagged slot with the third buffer and without; the walks of
the streaming operators and of DUGKS on more such grids; the 32 x 32 tiles and the depths beyond
8; and FP32 BGK tiles in FP64 arithmetic against FP64."""
from __future__ import annotations

import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu

MODELS = ["bgk", "trt", "rr", "bgk_split"]
OMEGA = 1.0 / (3 * 0.004 + 0.5)


def fields(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return (np.asfortranarray(1 + 0.01 * rng.standard_normal((ny, nx))),
            np.asfortranarray(0.05 * rng.standard_normal((ny, nx))),
            np.asfortranarray(0.05 * rng.standard_normal((ny, nx))))


def lattice(P, storage, nx, ny, omega=OMEGA):
    lat = P.Lattice(nx, ny, 2, storage)
    lat.set_params(omega, 0.25)
    lat.equilibrium_init(0, *fields(nx, ny, 1))
    return lat


def walk(P, storage, model, nx, ny, steps, depth, segments, third=True):
    lat = lattice(P, storage, nx, ny)
    lat.set_steps_per_launch(model, depth)
    lat.set_pass_segments(segments)
    lat.set_pass_lag_buffer(third)
    i, n = lat.run(model, steps, 0, 1)
    out = lat.download_f(i)[:ny], lat.download_f(n)[:ny]
    lat.close()
    return (i, n), out


@pytest.mark.parametrize("nx,ny", [(200, 130), (64, 64), (5, 3), (1, 7), (70, 1)])
@pytest.mark.parametrize("model", MODELS)
def test_fp64_equals_single_steps(P, gpu, model, nx, ny):
    for steps in (11, 8):
        ids, want = walk(P, "f64", model, nx, ny, steps, 1, 0)
        for depth in range(2, 9):
            for segments, third in ((1, True), (3, True), (3, False)):
                what = f"walk {model} {nx}x{ny} {steps} steps by {depth}, {segments} segments"
                print("case", what, flush=True)
                got_ids, got = walk(P, "f64", model, nx, ny, steps, depth, segments, third)
                assert got_ids == ids
                for a, w in zip(got, want):
                    np.testing.assert_array_equal(a, w, err_msg=what)


# populations after 10 steps (deviations to 0.15): FP64 and FP32 rounding with FMAs placed
# differently, about 30 roundings per step of at most 2^-3 x 2^-53 / 2^-24; FP16 (scale 2^10)
# rounds them to 2^-13 each time that a state is stored, which single steps do 10 times
TOL = {"f64s": 1e-14, "f32s": 1e-6, "f16s": 6e-4}


@pytest.mark.parametrize("storage", list(TOL))
@pytest.mark.parametrize("model", MODELS)
def test_shifted_matches_single_steps(P, gpu, storage, model):
    nx, ny, steps = 150, 100, 10
    ids, want = walk(P, storage, model, nx, ny, steps, 1, 0)
    for depth in range(2, 9):
        for segments in (2, 5):
            print(f"case walk {storage} {model} by {depth}, {segments} segments", flush=True)
            got_ids, got = walk(P, storage, model, nx, ny, steps, depth, segments)
            assert got_ids == ids
            for a, w in zip(got, want):
                np.testing.assert_allclose(a, w, rtol=0, atol=TOL[storage])


@pytest.mark.parametrize("third", [True, False])
@pytest.mark.parametrize("depth", [2, 3, 4, 8])
def test_step_counts(P, gpu, depth, third):
    nx, ny = 96, 80
    for steps in range(1, 21):
        ids, want = walk(P, "f64", "bgk", nx, ny, steps, 1, 0)
        got_ids, got = walk(P, "f64", "bgk", nx, ny, steps, depth, 4, third)
        assert got_ids == ids, steps
        for a, w in zip(got, want):
            np.testing.assert_array_equal(a, w, err_msg=str(steps))


# ragged sides just beyond the tiles' limits, and one whose segments are all alike (the pass with
# the lagged state then has a barrier per column)
@pytest.mark.parametrize("model,nx,ny", [("bgk", 1301, 1103), ("bgk_split", 1301, 1103),
                                         ("trt", 901, 841), ("trt", 1024, 1008),
                                         ("rr", 1361, 1327)])
def test_automatic_split(P, gpu, oracle, model, nx, ny):
    print(f"case walk auto {model} {nx}x{ny}", flush=True)
    steps = 15
    lat = lattice(P, "f64", nx, ny)
    lat.set_run_timing(True)
    i, n = lat.run(model, steps, 0, 1)
    assert [d for d, _ in lat.run_launch_times()] == [7, 8]  # tiles would share them otherwise
    fa, fb = po.new_f(nx, ny), po.new_f(nx, ny)
    oracle.set_pdf_to_equilibrium(nx, ny, *fields(nx, ny, 1), fa)
    latest, prev = oracle.run(model, nx, ny, fa, fb, steps, OMEGA, 0.25)
    np.testing.assert_array_equal(lat.download_f(i)[:ny], latest[:ny])
    np.testing.assert_array_equal(lat.download_f(n)[:ny], prev[:ny])


OPS = ["fvm_bardow", "fdm_bardow", "fdm_sofonea", "fdm_bardow_wls", "fdm_bardow_iso"]


@pytest.mark.parametrize("nx,ny", [(1009, 1013), (601, 1699), (3001, 341)])
@pytest.mark.parametrize("op", OPS)
def test_operator_walks(P, gpu, op, nx, ny):
    for model, steps, depth in (("bgk", 7, 0), ("trt", 4, 0), ("rr", 5, 2), ("bgk_split", 6, 3)):
        what = f"{op}+{model} {nx}x{ny} {steps} steps by {depth}"
        print("case walk", what, flush=True)
        lat, ref = lattice(P, "f64", nx, ny), lattice(P, "f64", nx, ny)
        lat.set_op_steps_per_pass(depth)
        ref.set_op_steps_per_pass(1)
        ids = lat.run_op(op, model, steps, 0, 1, 0.5)
        assert ids == ref.run_op(op, model, steps, 0, 1, 0.5)
        for b in ids:
            np.testing.assert_array_equal(lat.download_f(b)[:ny], ref.download_f(b)[:ny],
                                          err_msg=what)


@pytest.mark.parametrize("nx,ny,rates", [(709, 711, (1.75, 1.6)), (401, 1301, (1.75, 1.6)),
                                         (1009, 1013, (1.7, 1.7)), (601, 1699, (1.7, 1.7))])
def test_dugks_walks(P, gpu, nx, ny, rates):
    for steps in (1, 2, 5, 6):
        print(f"case walk dugks {nx}x{ny} {steps} steps", flush=True)
        lat, ref = lattice(P, "f64", nx, ny), lattice(P, "f64", nx, ny)
        ref.dugks_set_steps_per_pass(1)
        lat.dugks_step(0, 1, steps, 0.6, *rates)
        ref.dugks_step(0, 1, steps, 0.6, *rates)
        for b in (0, 1):
            np.testing.assert_array_equal(lat.download_f(b)[:ny], ref.download_f(b)[:ny])


@pytest.mark.parametrize("model", MODELS)
def test_tiles_of_32(P, gpu, oracle, model):
    """At the edges of the 32 x 32 tiles, and of the deepest ones of every shape."""
    for ns in (2, 5, 8, 9, 10, 11):
        shapes = [(32, 32)] if ns <= 8 else [(24, 24), (32, 32), (34, 32), (48, 46)]
        sizes = [(w - 2 * (ns - 1) + d, h - 2 * (ns - 1) + e) for w, h in shapes
                 for d, e in ((0, 0), (1, 0), (0, 1), (1, 1))]
        for nx, ny in sizes + [(2 * w, 3 * h) for w, h in sizes[:1]]:
            print(f"case tile {model} ns={ns} {nx}x{ny}", flush=True)
            lat = lattice(P, "f64", nx, ny)
            if ns <= 8:
                lat.set_steps_per_launch(model, ns)
            i, n = lat.run(model, ns, 0, 1)  # beyond 8 as the run chooses: up to 11 in one pass
            fa, fb = po.new_f(nx, ny), po.new_f(nx, ny)
            oracle.set_pdf_to_equilibrium(nx, ny, *fields(nx, ny, 1), fa)
            latest, prev = oracle.run(model, nx, ny, fa, fb, ns, OMEGA, 0.25)
            np.testing.assert_array_equal(lat.download_f(i)[:ny], latest[:ny])
            np.testing.assert_array_equal(lat.download_f(n)[:ny], prev[:ny])


@pytest.mark.parametrize("nx,ny", [(700, 640), (641, 701)])
def test_fp32_bgk_tiles_against_fp64(P, gpu, nx, ny):
    """Grids whose FP32 BGK tiles replace column walks: 300 steps of a Taylor-Green vortex against
    FP64.  Deviations of up to 2^-5 are rounded to half of 2^-28 once a step; a velocity sums
    six of them: 300 steps make a random walk of 300^0.5 x 2.6e-9, 5.5 times that among 4e5
    cells, 2.5e-7."""
    k = 2 * np.pi / max(nx, ny)
    x, y = (np.arange(nx) + 0.5)[None, :] * k, (np.arange(ny) + 0.5)[:, None] * k
    m = (np.ones((ny, nx)), -0.05 * np.cos(x) * np.sin(y), 0.05 * np.sin(x) * np.cos(y))
    u = {}
    for storage in ("f64", "f32s"):
        lat = P.Lattice(nx, ny, 2, storage)
        lat.set_params(1.0 / (3 * 0.03 + 0.5), 0.25)
        lat.equilibrium_init(0, *m)
        lat.set_run_timing(True)
        i, _ = lat.run("bgk", 300, 0, 1)
        u[storage] = np.stack(lat.macros(i)[1:])
    assert np.max(np.abs(u["f32s"] - u["f64"])) <= 2.5e-7
