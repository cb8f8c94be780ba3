"""Batch.macros against the same sums over Batch.download_f, bit for bit; batches in passes
held in LDS tiles against single steps, bit for bit (FP16: one step per pass; deeper passes
round less often)."""
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


@pytest.mark.parametrize("storage,model,per_pass", [("f64", "rr", 8), ("f64", "bgk", 2), ("f64s", "trt", 5),
                                                    ("f32s", "rr", 6), ("f32s", "trt", 7),
                                                    ("f16s", "trt", 2)])
def test_batch_tile_passes_equal_single_steps(P, gpu, storage, model, per_pass):
    """Step counts that split into passes of uneven depth, single steps among them; cases
    smaller than a tile's halo, at a tile's edge, and of several tiles, and resident ones."""
    sizes = [(1, 1), (5, 3), (34, 32), (35, 19), (130, 47), (20, 20), (257, 64)]
    rng = np.random.default_rng(5)
    fields = [tuple(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0))
              for nx, ny in sizes]

    def batch():
        b = P.Batch(sizes, storage, model)
        b.set_params([1.7] * len(sizes), [0.25] * len(sizes))
        for c, f in enumerate(fields):
            b.equilibrium_init(c, *f)
        return b

    for steps in (1, 2, per_pass + 1, 3 * per_pass):
        if storage == "f16s" and steps > 2:  # a pass of two steps rounds once
            continue
        print(f"case batch tiles {storage} {model} passes of {per_pass}, {steps} steps", flush=True)
        b, ref = batch(), batch()
        b.set_launch(128, 1, 400, 256)  # 20 x 20 and smaller run resident
        b.set_steps_per_pass(per_pass)
        b.run(steps)
        ref.run(steps, graph=False)
        for c in range(len(sizes)):
            np.testing.assert_array_equal(b.download_f(c), ref.download_f(c), err_msg=str(c))
