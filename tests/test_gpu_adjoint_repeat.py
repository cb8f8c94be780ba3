"""backward() more than once after one forward(): the same gradients each time, directly and
through autograd (retain_graph), and after a forward() of other fields."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fields(nx, ny, seed):
    import torch
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(np.ascontiguousarray(m + 0.03 * rng.standard_normal((nx, ny)))).cuda()
            for m in (1.0, 0.0, 0.0, 0.0, 0.0)]


@pytest.mark.parametrize("storage", ["f64", "f64s", "f32s"])
@pytest.mark.parametrize("steps,every", [(1, 1), (2, 1), (5, 2), (20, 5), (23, 10), (9, 9)])
def test_backward_repeats(P, gpu, steps, every, storage):
    import torch
    nx, ny = 61, 47
    print(f"case adjoint twice {storage} {steps} steps, every {every}", flush=True)
    eng = P.Adjoint(nx, ny, steps, every, storage)
    for seed in (1, 2):
        f = fields(nx, ny, seed)
        eng.forward(f[0], f[1], f[2], 1.6, f[3], f[4])
        first = eng.backward()
        for _ in range(2):
            again = eng.backward()
            for a, b in zip(first[:3], again[:3]):
                assert torch.equal(a, b)
            assert first[3] == again[3]
    eng.close()


def test_retain_graph(P, gpu):
    import torch
    nx, ny = 40, 33
    f = fields(nx, ny, 3)
    eng = P.Adjoint(nx, ny, 12, 4, "f64")
    ux, uy = f[1].requires_grad_(True), f[2].requires_grad_(True)
    tau = torch.tensor(0.7, dtype=torch.float64, requires_grad=True)
    loss = P.velocity_misfit(ux, uy, tau, f[3], f[4], eng)
    loss.backward(retain_graph=True)
    once = [v.grad.clone() for v in (ux, uy, tau)]
    loss.backward()
    for v, g in zip((ux, uy, tau), once):
        assert torch.equal(v.grad, 2 * g)


def test_backward_needs_a_forward(P, gpu):
    eng = P.Adjoint(16, 16, 4, 2, "f64")
    with pytest.raises(P.PlbmError, match="forward"):
        eng.backward()
