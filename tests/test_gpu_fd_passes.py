"""Passes of the streaming operators and of DUGKS in LDS tiles and in column walks, against
single steps bit for bit: tile edges, ragged and tiny grids, automatic depths, populations
that are not finite or close to overflow (whose zero terms then count), and capture."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OPS = ["fvm_bardow", "fdm_bardow", "fdm_sofonea", "fdm_bardow_wls", "fdm_bardow_wls_gauss_v1",
       "fdm_bardow_iso"]
# tiles of 24 x 24 and 34 x 33 less 2 ns; one grid above the tiles' 10^6 cells
EDGES = [(24 - 8, 24 - 8), (24 - 7, 24 - 8), (34 - 8, 33 - 7), (35, 19), (5, 3), (1, 9), (130, 1)]
LARGE = (1200, 841)


def lattice(P, nx, ny, poison=None, seed=1):
    rng = np.random.default_rng(seed)
    lat = P.Lattice(nx, ny, 2, "f64")
    lat.set_params(1.0 / (3 * 0.02 + 0.5), 0.25)
    lat.equilibrium_init(0, *(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)))
    if poison is not None:
        f = lat.download_f(0)
        for (y, x, q), v in poison.items():
            f[y % ny, x % nx, q] = v
        lat.upload_f(0, f)
    return lat


def compare(lat, ref, ids, ref_ids, ny, what):
    assert ids == ref_ids, what
    for i in ids:
        np.testing.assert_array_equal(lat.download_f(i)[:ny], ref.download_f(i)[:ny], err_msg=what)


@pytest.mark.parametrize("model", ["bgk", "trt", "rr", "bgk_split"])
@pytest.mark.parametrize("op", OPS)
def test_operator_passes_at_tile_edges(P, gpu, op, model):
    for nx, ny in EDGES:
        for depth, steps in ((0, 11), (2, 4), (3, 7)):
            what = f"case {op}+{model} {nx}x{ny} passes of {depth}, {steps} steps"
            print(what, flush=True)
            lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
            lat.set_op_steps_per_pass(depth)
            ref.set_op_steps_per_pass(1)
            compare(lat, ref, lat.run_op(op, model, steps, 0, 1, 0.7),
                    ref.run_op(op, model, steps, 0, 1, 0.7), ny, what)


@pytest.mark.parametrize("op", OPS)
def test_operator_walks(P, gpu, op):
    nx, ny = LARGE
    for steps in (2, 9):  # one pass of 2; 2 + 3 + 4, the last with the lagged state
        print(f"case walk {op} {nx}x{ny} {steps} steps", flush=True)
        lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
        ref.set_op_steps_per_pass(1)
        compare(lat, ref, lat.run_op(op, "rr", steps, 0, 1, 0.4),
                ref.run_op(op, "rr", steps, 0, 1, 0.4), ny, f"{op} {steps}")


POISON = {"inf": np.inf, "-inf": -np.inf, "nan": np.nan, "large": 1e303, "lowest": -1.7e308,
          "tiny": 5e-324}


@pytest.mark.parametrize("value", list(POISON))
@pytest.mark.parametrize("nx,ny", [(70, 45), LARGE])
@pytest.mark.parametrize("op", ["fvm_bardow", "fdm_bardow", "fdm_sofonea", "fdm_bardow_wls"])
def test_operator_passes_of_values_out_of_range(P, gpu, op, nx, ny, value):
    """Single populations replaced in the interior, at a corner and at a tile's or band's
    edge: the same cells become the same numbers, infinities and NaNs."""
    poison = {(20, 30, 1): POISON[value], (0, 0, 2): POISON[value], (ny - 1, 33, 5): POISON[value]}
    what = f"case {op} {value} {nx}x{ny}"
    print(what, flush=True)
    lat, ref = lattice(P, nx, ny, poison), lattice(P, nx, ny, poison)
    ref.set_op_steps_per_pass(1)
    compare(lat, ref, lat.run_op(op, "bgk", 5, 0, 1, 0.4), ref.run_op(op, "bgk", 5, 0, 1, 0.4),
            ny, what)


def test_operator_runs_under_capture(P, gpu):
    """Small grids keep single steps while captured, so that replays continue."""
    import torch
    nx, ny, steps = 96, 80, 6
    lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
    ref.set_op_steps_per_pass(1)
    s = torch.cuda.Stream()
    lat.set_stream(s.cuda_stream)
    lat.run_op("fvm_bardow", "trt", steps, 0, 1, 0.5)
    ref.run_op("fvm_bardow", "trt", steps, 0, 1, 0.5)
    lat.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        assert lat.run_op("fvm_bardow", "trt", steps, 0, 1, 0.5) == (0, 1)
    for replay in range(3):
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        ref.run_op("fvm_bardow", "trt", steps, 0, 1, 0.5)
        compare(lat, ref, (0, 1), (0, 1), ny, f"replay {replay}")


RATES = {"equal": (0.4, 1.7, 1.7), "unequal": (0.7, 1.75, 1.6)}
# 24 x 24 and 34 x 33 tiles; walks above 10^6 cells, or 5 10^5 at unequal rates
DUGKS_GRIDS = EDGES + [(900, 613), LARGE]


@pytest.mark.parametrize("rates", list(RATES))
@pytest.mark.parametrize("nx,ny", DUGKS_GRIDS)
def test_dugks_passes(P, gpu, nx, ny, rates):
    """Automatic runs, whose last pass stores the half-collided state as well, and passes of a
    chosen depth against the collide + flux pair."""
    for depth, steps in ((0, 1), (0, 2), (0, 11), (2, 6), (3, 8)):
        what = f"case dugks {rates} {nx}x{ny} passes of {depth}, {steps} steps"
        print(what, flush=True)
        lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
        lat.dugks_set_steps_per_pass(depth)
        ref.dugks_set_steps_per_pass(1)
        lat.dugks_step(0, 1, steps, *RATES[rates])
        ref.dugks_step(0, 1, steps, *RATES[rates])
        compare(lat, ref, (0, 1), (0, 1), ny, what)


@pytest.mark.parametrize("value", list(POISON))
@pytest.mark.parametrize("rates", list(RATES))
@pytest.mark.parametrize("nx,ny", [(70, 45), LARGE])
def test_dugks_passes_of_values_out_of_range(P, gpu, nx, ny, rates, value):
    poison = {(20, 30, 1): POISON[value], (0, 0, 2): POISON[value], (ny - 1, 33, 5): POISON[value]}
    what = f"case dugks {rates} {value} {nx}x{ny}"
    print(what, flush=True)
    lat, ref = lattice(P, nx, ny, poison), lattice(P, nx, ny, poison)
    ref.dugks_set_steps_per_pass(1)
    lat.dugks_step(0, 1, 5, *RATES[rates])
    ref.dugks_step(0, 1, 5, *RATES[rates])
    compare(lat, ref, (0, 1), (0, 1), ny, what)


@pytest.mark.parametrize("rates", list(RATES))
def test_dugks_under_capture_and_without_third_buffer(P, gpu, rates):
    import torch
    nx, ny, steps = 96, 80, 6
    lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
    ref.dugks_set_steps_per_pass(1)
    s = torch.cuda.Stream()
    lat.set_stream(s.cuda_stream)
    lat.dugks_step(0, 1, steps, *RATES[rates])
    ref.dugks_step(0, 1, steps, *RATES[rates])
    lat.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        lat.dugks_step(0, 1, steps, *RATES[rates])
    for replay in range(3):
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        ref.dugks_step(0, 1, steps, *RATES[rates])
        compare(lat, ref, (0, 1), (0, 1), ny, f"replay {replay}")
    lat.set_pass_lag_buffer(False)
    lat.dugks_step(0, 1, 7, *RATES[rates])
    ref.dugks_step(0, 1, 7, *RATES[rates])
    compare(lat, ref, (0, 1), (0, 1), ny, "two buffers")
