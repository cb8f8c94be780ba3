"""Device memory of an adjoint beside its states: the omega sensitivity's partial sums are few
whatever the grid's shape (many tiles of few cells), and their total is right."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,storage", [(1, 400000, "f64"), (1, 400000, "f32s"),
                                           (1000, 1000, "f64")])
def test_memory_of_an_adjoint(P, gpu, nx, ny, storage):
    import torch
    print(f"case adjoint memory {nx}x{ny} {storage}", flush=True)
    P.Adjoint(8, 8, 2, 1, storage).close()  # what a first use loads is not the adjoint's
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    eng = P.Adjoint(nx, ny, 2, 1, storage)
    used = before - torch.cuda.mem_get_info()[0]
    state = 9 * nx * ((ny + 63) // 64 * 64)
    # two buffers, two checkpoints and a segment of one state in the storage, the adjoint states
    # in FP64 (8-byte storages: one beside the two buffers), and allocations rounded up to 2 MiB
    want = 5 * 8 * state + 8 * state if storage == "f64" else 5 * 4 * state + 3 * 8 * state
    assert used <= 1.05 * want + 10 * 2 ** 21
    eng.close()


def test_total_over_many_tiles(P, gpu):
    """A field that repeats along the columns: the sensitivity as often as it repeats."""
    import torch
    rng = np.random.default_rng(4)
    f = [m + 0.03 * rng.standard_normal((2, 24)) for m in (1.0, 0.0, 0.0, 0.0, 0.0)]
    out = []
    for times in (1, 4000):
        t = [torch.from_numpy(np.ascontiguousarray(np.tile(a, (1, times)))).cuda() for a in f]
        eng = P.Adjoint(2, 24 * times, 9, 4, "f64")
        loss = eng.forward(t[0], t[1], t[2], 1.6, t[3], t[4])
        out.append((loss / times, eng.backward()[3] / times))
        eng.close()
    assert out[1] == pytest.approx(out[0], rel=1e-12)
