"""Fields read back through pinned memory (small ones, two sizes of it) and by copies, against
the fields on the device; update_macros into the grid's planes and into a replaced array."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one column, odd column counts; 2^20 and 5 2^19 bytes of three FP64 fields and beyond
SIZES = [(1, 1), (1, 300), (2, 1), (3, 77), (128, 341), (128, 342), (320, 341), (320, 342)]


def moments(nx, ny, seed=2):
    rng = np.random.default_rng(seed)
    return [c + 0.03 * rng.standard_normal((ny, nx)) for c in (1.0, 0.0, 0.0)]


@pytest.mark.parametrize("storage", ["f64", "f16s"])
def test_macros(P, gpu, storage):
    import torch
    for nx, ny in SIZES:
        print(f"case macros {nx}x{ny} {storage}", flush=True)
        lat = P.Lattice(nx, ny, 2, storage)
        lat.set_params(1.7, 0.25)
        lat.equilibrium_init(0, *moments(nx, ny))
        dev = torch.empty(3, nx, ny, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        lat.macros_dev(0, *(d.data_ptr() for d in dev))
        lat.sync()
        for _ in range(2):
            for a, d in zip(lat.macros(0), dev.cpu().numpy()):
                np.testing.assert_array_equal(a, d.T)


def test_batch_macros(P, gpu):
    """Cases of all sizes in one batch, the larger pinned size after the smaller and before."""
    b = P.Batch(SIZES, "f64", "bgk")
    b.set_params([1.7] * len(SIZES), [0.25] * len(SIZES))
    want = []
    for c, (nx, ny) in enumerate(SIZES):
        m = moments(nx, ny, c)
        b.equilibrium_init(c, *m)
        lat = P.Lattice(nx, ny, 2, "f64")
        lat.equilibrium_init(0, *m)
        want.append(lat.macros(0))
    for order in (range(len(SIZES)), reversed(range(len(SIZES)))):
        for c in order:
            # rounding of two orders of summation
            for a, w in zip(b.macros(c), want[c]):
                np.testing.assert_allclose(a, w, rtol=0, atol=1e-14)


def test_update_macros(P, gpu):
    nx, ny = 33, 21
    fields = []
    for layout in ("planes", "replaced"):
        g = P.alloc_grid(nx, ny, log=False)
        P.set_properties(g, 0.02, 1.0, 0.25)
        g.streaming, g.collision = P.lbm_stream, P.collide_bgk
        for to, m in zip((g.rho, g.ux, g.uy), moments(nx, ny)):
            to[:] = m
        P.set_pdf_to_equilibrium(g)
        if layout == "replaced":
            g.mf = np.zeros((ny, nx, 3))  # C order: no plane is contiguous
        for _ in range(3):
            P.perform_step(g)
        P.update_macros(g)
        fields.append(np.array(g.mf))
        P.dealloc_grid(g)
    assert np.ptp(fields[0][:, :, 1]) > 0
    np.testing.assert_array_equal(fields[0], fields[1])
