"""Autotuning on grids that run in tiles: a tuned lattice keeps the automatic plan (depths to 11,
chosen for the run's length) and its results, and what was tuned under another work split is not
taken over."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def lattice(P, storage, nx, ny):
    rng = np.random.default_rng(nx + ny)
    lat = P.Lattice(nx, ny, 2, storage)
    lat.set_params(1.7, 0.25)
    lat.equilibrium_init(0, *(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)))
    lat.set_run_timing(True)
    return lat


def depths(lat):
    return [d for d, _ in lat.run_launch_times()]


@pytest.mark.parametrize("model", ["bgk", "trt", "rr"])
@pytest.mark.parametrize("storage", ["f64", "f32s", "f16s"])
def test_tuned_runs_as_untuned(P, gpu, storage, model):
    for nx, ny, steps in ((64, 64, 50), (131, 90, 23)):
        print(f"case autotune {storage} {model} {nx}x{ny}", flush=True)
        lat, ref = lattice(P, storage, nx, ny), lattice(P, storage, nx, ny)
        assert lat.autotune(model, 0, reps=3) > 0
        ids = lat.run(model, steps, 0, 1)
        assert ids == ref.run(model, steps, 0, 1)
        assert depths(lat) == depths(ref)
        assert max(depths(ref)) > 8 or storage != "f64" or nx > 64
        for b in (0, 1):
            np.testing.assert_array_equal(lat.download_f(b), ref.download_f(b))


def test_tuned_under_another_split(P, gpu):
    """One segment per band walks columns; a later lattice of the same size does not."""
    first, lat, ref = (lattice(P, "f64", 72, 72) for _ in range(3))
    first.set_pass_segments(1)
    first.autotune("trt", 0, reps=2)
    lat.autotune("trt", 0, reps=2)
    for l in (lat, ref):
        l.run("trt", 22, 0, 1)
    assert depths(lat) == depths(ref) and max(depths(lat)) > 1
