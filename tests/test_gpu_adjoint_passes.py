"""Reverse sweep in LDS tiles: gradients against PyTorch autograd of the same BGK steps in FP64
(tile edges, ragged and tiny grids, checkpoint intervals), and the 64-bit offsets."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]
W = [4 / 9] + [1 / 9] * 4 + [1 / 36] * 4


def fields(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return [1 + 0.02 * rng.standard_normal((nx, ny))] + \
        [0.05 * rng.standard_normal((nx, ny)) for _ in range(4)]


def equilibrium(rho, ux, uy):
    u2 = ux * ux + uy * uy
    return [w * rho * (1 + 3 * (a * ux + b * uy) + 4.5 * (a * ux + b * uy) ** 2 - 1.5 * u2)
            for w, (a, b) in zip(W, C)]


def reference(fs, steps, omega):
    """Loss and its gradients in rho0, ux0, uy0, omega, on the CPU."""
    import torch
    rho0, ux0, uy0, uxt, uyt = (torch.from_numpy(f) for f in fs)
    var = [v.requires_grad_(True) for v in (rho0, ux0, uy0)]
    om = torch.tensor(omega, dtype=torch.float64, requires_grad=True)

    def moments(f):
        rho = sum(f)
        return (rho, sum(a * v for v, (a, _) in zip(f, C)) / rho,
                sum(b * v for v, (_, b) in zip(f, C)) / rho)
    f = equilibrium(*var)
    for _ in range(steps):
        g = [torch.roll(v, c, (0, 1)) for v, c in zip(f, C)]
        f = [(1 - om) * a + om * e for a, e in zip(g, equilibrium(*moments(g)))]
    _, ux, uy = moments(f)
    loss = 0.5 * ((ux - uxt) ** 2 + (uy - uyt) ** 2).sum()
    loss.backward()
    return float(loss.detach()), [v.grad.numpy() for v in var], float(om.grad)


def engine(P, fs, steps, every, omega, storage):
    import torch
    nx, ny = fs[0].shape
    t = [torch.from_numpy(np.ascontiguousarray(f)).cuda() for f in fs]
    eng = P.Adjoint(nx, ny, steps, every, storage)
    loss = eng.forward(t[0], t[1], t[2], omega, t[3], t[4])
    *g, gom = eng.backward()
    out = loss, [v.cpu().numpy() for v in g], gom
    eng.close()
    return out


# Rounding: about 10 operations on the way of a value through a step, 20 steps, 2^-53 each of
# values up to 1 against gradients of 0.1: below 1e-12.  FP32 storage rounds deviations of 0.1
# to 6e-9 each step, against velocities of 0.05.
@pytest.mark.parametrize("storage,tol", [("f64", 1e-11), ("f64s", 1e-11), ("f32s", 5e-5)])
@pytest.mark.parametrize("nx,ny", [(24, 24), (25, 23), (10, 11), (1, 9), (9, 1), (3, 2), (130, 47),
                                   (300, 17)])
def test_gradients_against_autograd(P, gpu, nx, ny, storage, tol):
    for steps, every in ((1, 1), (2, 5), (9, 4), (20, 20), (17, 8)):
        print(f"case adjoint {storage} {nx}x{ny} {steps} steps, every {every}", flush=True)
        fs = fields(nx, ny, nx + 10 * steps)
        loss, grads, gom = engine(P, fs, steps, every, 1.6, storage)
        ref_loss, ref_grads, ref_gom = reference(fs, steps, 1.6)
        assert abs(loss - ref_loss) <= tol * ref_loss
        for g, r in zip(grads, ref_grads):
            assert np.max(np.abs(g - r)) <= tol * np.max(np.abs(r))
        # a sum over cells of terms of either sign: against the velocities' gradients
        scale = nx * ny * max(np.max(np.abs(r)) for r in ref_grads) * 0.1
        assert abs(gom - ref_gom) <= tol * scale


def test_offsets_beyond_32_bits(P, gpu):
    """Columns too long for 32-bit offsets give the bits of the short ones that they repeat."""
    nx, ny, times = 4, 24, 10000
    fs = fields(nx, ny, 3)
    print(f"case adjoint {nx}x{ny * times}", flush=True)
    loss, grads, gom = engine(P, fs, 11, 6, 1.6, "f64")
    loss2, grads2, gom2 = engine(P, [np.tile(f, (1, times)) for f in fs], 11, 6, 1.6, "f64")
    for g, g2 in zip(grads, grads2):
        np.testing.assert_array_equal(np.tile(g, (1, times)), g2)
    assert gom2 == pytest.approx(gom * times, rel=1e-12)
    assert loss2 == pytest.approx(loss * times, rel=1e-12)
