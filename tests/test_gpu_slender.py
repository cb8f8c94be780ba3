"""Long grids of few columns keep single steps and column walks (their tiles would be mostly halo):
the routes at both sides of the rules, and their results against single steps."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lattice(P, nx, ny, storage="f64"):
    rng = np.random.default_rng(nx)
    lat = P.Lattice(nx, ny, 2, storage)
    lat.set_params(1.7, 0.25)
    lat.equilibrium_init(0, *(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)))
    return lat


def same(lat, ref, ids):
    for b in ids:
        np.testing.assert_array_equal(lat.download_f(b), ref.download_f(b))


# columns, rows, whether plbm_run walks them in passes of 8
@pytest.mark.parametrize("nx,ny,storage,walks", [
    (1, 32768, "f64", False), (1, 32769, "f64", True), (4, 33000, "f64", True),
    (5, 33000, "f64", False), (8, 33000, "f32s", True), (9, 33000, "f32s", False)])
def test_runs(P, gpu, nx, ny, storage, walks):
    print(f"case slender run {nx}x{ny} {storage}", flush=True)
    lat, ref = lattice(P, nx, ny, storage), lattice(P, nx, ny, storage)
    ref.set_steps_per_launch("trt", 1)
    lat.set_run_timing(True)
    ids = lat.run("trt", 24, 0, 1)
    assert ids == ref.run("trt", 24, 0, 1)
    assert ([d for d, _ in lat.run_launch_times()] == [8, 8, 8]) == walks
    if storage == "f64":
        same(lat, ref, ids)


@pytest.mark.parametrize("nx,ny,one,two", [  # single steps at equal rates, at unequal ones
    (1, 16384, False, False), (1, 16385, True, True), (2, 24000, False, True),
    (2, 24577, True, True), (4, 40961, True, True), (5, 50000, False, False)])
def test_operators_and_dugks(P, gpu, nx, ny, one, two):
    print(f"case slender operators {nx}x{ny}", flush=True)
    lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
    ref.set_op_steps_per_pass(1)
    ref.dugks_set_steps_per_pass(1)
    assert (lat.get_op_steps_per_pass() == 1) == one
    assert (lat.dugks_get_steps_per_pass() == 1) == one
    ids = lat.run_op("fvm_bardow", "bgk", 8, 0, 1, 0.4)
    assert ids == ref.run_op("fvm_bardow", "bgk", 8, 0, 1, 0.4)
    same(lat, ref, ids)
    for rates in ((1.7, 1.7), (1.75, 1.6)):
        before = {lat.buffer_ptr(0), lat.buffer_ptr(1)}
        lat.dugks_step(0, 1, 4, 0.4, *rates)
        ref.dugks_step(0, 1, 4, 0.4, *rates)
        same(lat, ref, (0, 1))
        # single steps stay in the two slots; a tile pass takes the third buffer in turn
        single = one if rates[0] == rates[1] else two
        assert (before == {lat.buffer_ptr(0), lat.buffer_ptr(1)}) == single
