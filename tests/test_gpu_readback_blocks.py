"""Small fields read back through the process's two pinned blocks: by copies until a block would
have paid, then through it, from several lattices, threads and streams, after the blocks were
given back with the last lattice, and up to their sizes, against the fields on the device."""
from __future__ import annotations

import gc
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# columns x rows; 2^20 and 5 2^19 bytes of three FP64 fields and just beyond
SIZES = [(1, 1), (2, 7), (3, 1), (1, 43690), (128, 341), (1, 43691), (128, 342), (320, 341),
         (1, 109226), (320, 342), (7, 10000), (5000, 20)]


def moments(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return [c + 0.03 * rng.standard_normal((ny, nx)) for c in (1.0, 0.0, 0.0)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_reads(P, gpu, nx, ny):
    import torch
    print(f"case read-back {nx}x{ny}", flush=True)
    gc.collect()
    lat = P.Lattice(nx, ny, 2, "f64")
    lat.set_params(1.7, 0.25)
    dev = torch.empty(3, nx, ny, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for read in range(14):  # other fields each time
        lat.equilibrium_init(0, *moments(nx, ny, read))
        lat.macros_dev(0, *(d.data_ptr() for d in dev))
        lat.sync()
        for a, d in zip(lat.macros(0), dev.cpu().numpy()):
            np.testing.assert_array_equal(a, d.T, err_msg=f"read {read}")
    lat.close()


@pytest.mark.parametrize("nx,ny", [(64, 48), (300, 260)])
def test_reads_of_several_threads(P, gpu, nx, ny):
    print(f"case read-back in threads {nx}x{ny}", flush=True)
    lats, want, wrong = [], [], []
    for k in range(4):
        lat = P.Lattice(nx, ny, 2, "f64")
        lat.set_params(1.7, 0.25)
        lat.equilibrium_init(0, *moments(nx, ny, k))
        lat.sync()
        lats.append(lat)
        want.append(np.stack(lat.macros(0)))

    def read(k):
        for _ in range(30):
            if not np.array_equal(np.stack(lats[k].macros(0)), want[k]):
                wrong.append(k)
    threads = [threading.Thread(target=read, args=(k,)) for k in range(len(lats))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for k in range(1, 4):
        assert not np.array_equal(want[0], want[k])
