"""What the getters of a pass depth report can be set again, on every kind of grid (tiles,
column walks, single steps), and leaves the results as they are."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(64, 64), (300, 200), (1200, 900)])
def test_read_depth_can_be_set(P, gpu, nx, ny):
    print(f"case depth settings {nx}x{ny}", flush=True)
    rng = np.random.default_rng(1)
    m = [c + 0.02 * rng.standard_normal((ny, nx)) for c in (1.0, 0.0, 0.0)]
    out = []
    for restore in (False, True):
        lat = P.Lattice(nx, ny, 2, "f64")
        lat.set_params(1.7, 0.25)
        lat.equilibrium_init(0, *m)
        if restore:
            op, dugks, run = (lat.get_op_steps_per_pass(), lat.dugks_get_steps_per_pass(),
                              lat.get_steps_per_launch("trt"))
            lat.set_op_steps_per_pass(1)
            lat.dugks_set_steps_per_pass(1)
            lat.set_steps_per_launch("trt", 1)
            lat.set_op_steps_per_pass(op)
            lat.dugks_set_steps_per_pass(dugks)
            lat.set_steps_per_launch("trt", run)
            assert (lat.get_op_steps_per_pass(), lat.dugks_get_steps_per_pass(),
                    lat.get_steps_per_launch("trt")) == (op, dugks, run)
        i, n = lat.run_op("fvm_bardow", "trt", 7, 0, 1, 0.5)
        i, n = lat.run("trt", 9, i, n)
        lat.dugks_step(i, n, 8, 0.4, 1.7, 1.7)
        out.append((i, n, lat.download_f(i), lat.download_f(n)))
    assert out[0][:2] == out[1][:2]
    for a, b in zip(out[0][2:], out[1][2:]):
        np.testing.assert_array_equal(a, b)
