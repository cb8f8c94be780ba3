"""FP16 storage computes in FP32: a step from populations that both reduced storages hold
exactly is the FP32-storage step rounded to FP16 (scale 2^10), bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

W = np.array([4 / 9] + [1 / 9] * 4 + [1 / 36] * 4)
SCALE = 1024.0


@pytest.mark.parametrize("model", ["bgk", "bgk_split"])
@pytest.mark.parametrize("nx,ny,omega", [(130, 97, 1.7), (64, 64, 1.97), (7, 300, 0.6)])
def test_step_is_the_fp32_step_rounded(P, gpu, nx, ny, omega, model):
    print(f"case fp16 step {model} {nx}x{ny}", flush=True)
    rng = np.random.default_rng(nx + ny)
    dev = (rng.uniform(-0.02, 0.02, (ny, nx, 9)) * SCALE).astype(np.float16) / SCALE
    out = {}
    for storage in ("f32s", "f16s"):
        lat = P.Lattice(nx, ny, 2, storage)
        lat.set_params(omega, 0.25)
        lat.upload_f(0, np.asfortranarray(dev + W))
        # the weights added in FP64 and taken off again leave the stored values recognisable
        np.testing.assert_allclose(lat.download_f(0)[:ny] - W, dev, rtol=0, atol=1e-15)
        lat.step(model, 0, 1)
        out[storage] = (lat.download_f(1)[:ny] - W) * SCALE
    np.testing.assert_array_equal(out["f16s"].astype(np.float16),
                                  out["f32s"].astype(np.float32).astype(np.float16))
