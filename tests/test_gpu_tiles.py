"""Tile passes (LDS, small and medium grids): at the edges of the three tile shapes and with
grids smaller than a tile's halo, every depth, against the oracle bit for bit in FP64 and
against single steps bit for bit in the other storages (FP16 rounding every level, as the
automatic depth does where single steps were the choice); and the automatic depth while the
stream is captured."""
from __future__ import annotations

import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu

OMEGA = 1.0 / (3 * 0.004 + 0.5)
# columns x rows of the shapes at level 1; a tile of ns steps is 2 (ns - 1) smaller
SHAPES = [(24, 24), (34, 32), (48, 46)]


def fields(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return (np.asfortranarray(1 + 0.01 * rng.standard_normal((ny, nx))),
            np.asfortranarray(0.05 * rng.standard_normal((ny, nx))),
            np.asfortranarray(0.05 * rng.standard_normal((ny, nx))))


def lattice(P, storage, nx, ny):
    lat = P.Lattice(nx, ny, 2, storage)
    lat.set_params(OMEGA, 0.25)
    lat.equilibrium_init(0, *fields(nx, ny, 1))
    return lat


@pytest.mark.parametrize("ns", range(2, 9))
@pytest.mark.parametrize("model", ["bgk", "trt", "rr", "bgk_split"])
def test_tile_edges_fp64(P, gpu, oracle, model, ns):
    sizes = [(w - 2 * (ns - 1) + d, h - 2 * (ns - 1) + e) for w, h in SHAPES
             for d, e in ((0, 0), (1, 0), (0, 1))]
    for nx, ny in sizes + [(1, 1), (2, 9), (97, 3)]:
        print(f"case tile {model} ns={ns} {nx}x{ny}", flush=True)
        lat = lattice(P, "f64", nx, ny)
        lat.set_steps_per_launch(model, ns)
        i, n = lat.run(model, 2 * ns, 0, 1)
        fa, fb = po.new_f(nx, ny), po.new_f(nx, ny)
        oracle.set_pdf_to_equilibrium(nx, ny, *fields(nx, ny, 1), fa)
        latest, prev = oracle.run(model, nx, ny, fa, fb, 2 * ns, OMEGA, 0.25)
        np.testing.assert_array_equal(lat.download_f(i)[:ny], latest[:ny])
        np.testing.assert_array_equal(lat.download_f(n)[:ny], prev[:ny])


@pytest.mark.parametrize("model", ["bgk", "trt", "rr"])
@pytest.mark.parametrize("storage", ["f64", "f64s", "f32s", "f16s"])
def test_automatic_depth_equals_single_steps(P, gpu, storage, model):
    """Grids on which single steps were the automatic choice: their results, both slots."""
    for nx, ny, steps in ((64, 64, 50), (201, 77, 9), (5, 3, 11), (320, 320, 2)):
        print(f"case tile auto {storage} {model} {nx}x{ny}", flush=True)
        lat, ref = lattice(P, storage, nx, ny), lattice(P, storage, nx, ny)
        ref.set_steps_per_launch(model, 1)
        lat.set_run_timing(True)
        i, n = lat.run(model, steps, 0, 1)
        assert max(d for d, _ in lat.run_launch_times()) > 1
        assert (i, n) == ref.run(model, steps, 0, 1)
        np.testing.assert_array_equal(lat.download_f(i), ref.download_f(i))
        np.testing.assert_array_equal(lat.download_f(n), ref.download_f(n))


@pytest.mark.parametrize("model", ["bgk", "trt", "rr"])
def test_automatic_depths_fp64(P, gpu, oracle, model):
    """The depths a run chooses, beyond 8 among them, at the edges of the one tile per compute
    unit that it chooses them for: oracle, bit for bit."""
    deepest = {}
    for nx, ny, steps in ((2, 3, 11), (32, 32, 23), (64, 64, 22), (65, 63, 12), (96, 97, 31),
                          (128, 128, 9), (129, 127, 19), (255, 256, 18), (257, 256, 10),
                          (320, 320, 7), (321, 319, 8), (400, 400, 11), (401, 399, 13)):
        print(f"case tile depth {model} {nx}x{ny} {steps} steps", flush=True)
        lat = lattice(P, "f64", nx, ny)
        lat.set_run_timing(True)
        i, n = lat.run(model, steps, 0, 1)
        deepest[nx, ny] = max(d for d, _ in lat.run_launch_times())
        fa, fb = po.new_f(nx, ny), po.new_f(nx, ny)
        oracle.set_pdf_to_equilibrium(nx, ny, *fields(nx, ny, 1), fa)
        latest, prev = oracle.run(model, nx, ny, fa, fb, steps, OMEGA, 0.25)
        np.testing.assert_array_equal(lat.download_f(i)[:ny], latest[:ny])
        np.testing.assert_array_equal(lat.download_f(n)[:ny], prev[:ny])
    assert deepest[64, 64] == 11 and deepest[2, 3] == 11


def test_automatic_depth_under_capture(P, gpu):
    """A captured run on a small grid stays in its two buffers, so that replays continue
    from each other; eager runs before and between do not disturb it."""
    import torch
    nx, ny, steps = 96, 80, 6
    lat, ref = lattice(P, "f64", nx, ny), lattice(P, "f64", nx, ny)
    ref.set_steps_per_launch("trt", 1)
    s = torch.cuda.Stream()
    lat.set_stream(s.cuda_stream)
    lat.run("trt", steps, 0, 1)
    lat.sync()
    ref.run("trt", steps, 0, 1)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        assert lat.run("trt", steps, 0, 1) == (0, 1)
    for replay in range(3):
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        ref.run("trt", steps, 0, 1)
        for b in (0, 1):
            np.testing.assert_array_equal(lat.download_f(b), ref.download_f(b), err_msg=str(replay))


@pytest.mark.parametrize("storage", ["f64", "f16s"])
@pytest.mark.parametrize("ny,block", [(1, 128), (127, 128), (128, 128), (129, 256), (256, 256),
                                      (257, 128), (384, 128), (385, 256), (1024, 256),
                                      (1025, 256)])
def test_single_step_workgroups(P, gpu, ny, block, storage):
    """Automatic workgroup sizes of single steps against 256 threads, bit for bit."""
    print(f"case single steps 7x{ny} {storage}", flush=True)
    rng = np.random.default_rng(ny)
    m = [c + 0.02 * rng.standard_normal((ny, 7)) for c in (1.0, 0.0, 0.0)]
    f = []
    for chosen in (None, 256):
        lat = P.Lattice(7, ny, 2, storage)
        lat.set_params(1.7, 0.25)
        assert lat.get_launch("rr") == (block, 1)
        if chosen:
            lat.set_launch("rr", chosen)
        lat.equilibrium_init(0, *m)
        lat.step("rr", 0, 1)
        f.append(lat.download_f(1)[:ny])
    np.testing.assert_array_equal(f[0], f[1])
