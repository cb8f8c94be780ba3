"""Batch.macros against the same sums over Batch.download_f, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f64s", "f32s", "f16s"])
@pytest.mark.parametrize("steps", [0, 3])  # the latest state in either buffer
def test_batch_macros_equal_downloaded_sums(P, gpu, storage, steps):
    sizes = [(5, 3), (64, 64), (33, 300), (1, 70)]
    b = P.Batch(sizes, storage, "trt")
    b.set_params([1.7] * len(sizes), [0.25] * len(sizes))
    rng = np.random.default_rng(3)
    for c, (nx, ny) in enumerate(sizes):
        b.equilibrium_init(c, *(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)))
    b.run(steps)
    for c, (nx, ny) in enumerate(sizes):
        print(f"case batch macros {storage} {nx}x{ny} after {steps}", flush=True)
        f = np.moveaxis(b.download_f(c)[:ny], 2, 0)
        rho = f[0] + (((f[5] + f[7]) + (f[6] + f[8])) + ((f[1] + f[3]) + (f[2] + f[4])))
        r, u, v = b.macros(c)
        np.testing.assert_array_equal(r, rho)
        np.testing.assert_array_equal(u, (((f[5] - f[7]) + (f[8] - f[6])) + (f[1] - f[3])) / rho)
        np.testing.assert_array_equal(v, (((f[5] - f[7]) + (f[6] - f[8])) + (f[2] - f[4])) / rho)
