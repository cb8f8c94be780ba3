"""Graphs captured from a lattice's calls, replayed between eager runs of the same lattice: the
slots' storage stays where the graph's addresses are, as if every run took single steps (small
grids), or the latest state does (larger grids, runs of an even number of passes)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DUGKS = (0.7, 1.75, 1.6)  # dt, the two rates


def lattice(P, nx, ny, storage="f64"):
    rng = np.random.default_rng(nx)
    lat = P.Lattice(nx, ny, 2, storage)
    lat.set_params(1.0 / (3 * 0.02 + 0.5), 0.25)
    lat.equilibrium_init(0, *(m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)))
    return lat


def single_steps(lat, storage="f64"):
    for model in ("bgk", "trt"):
        lat.set_steps_per_launch(model, 1)
    if storage == "f64":
        lat.set_op_steps_per_pass(1)
        lat.dugks_set_steps_per_pass(1)


def replay_between_runs(lat, ref, captured, eager, compare):
    """Two eager runs, the capture, then replays with eager runs between them; ref makes the
    same calls eagerly in single steps."""
    import torch
    s = torch.cuda.Stream()
    lat.set_stream(s.cuda_stream)
    for l in (lat, ref):
        eager(l)
        eager(l)
        l.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        captured(lat)
    for turn, what in enumerate("replay eager replay replay eager eager replay".split()):
        if what == "eager":
            eager(lat)
        else:
            with torch.cuda.stream(s):
                g.replay()
        torch.cuda.synchronize()
        (eager if what == "eager" else captured)(ref)
        compare(f"turn {turn}: {what}")


def both_slots(lat, ref):
    def compare(what):
        for b in (0, 1):
            np.testing.assert_array_equal(lat.download_f(b), ref.download_f(b), err_msg=what)
    return compare


def latest_slot(lat, ref):
    def compare(what):
        np.testing.assert_array_equal(np.stack(lat.macros(0)), np.stack(ref.macros(0)),
                                      err_msg=what)
    return compare


def run(model, steps):
    return lambda l: l.run(model, steps, 0, 1)


def two_steps(l):
    l.step("trt", 0, 1)
    l.step("trt", 1, 0)


def op(steps):
    return lambda l: l.run_op("fvm_bardow", "trt", steps, 0, 1, 0.5)


def dugks(l):
    l.dugks_step(0, 1, 6, *DUGKS)


def two_dugks_steps(l):
    l.dugks_step(0, 1, 1, *DUGKS)
    l.dugks_step(1, 0, 1, *DUGKS)


# what the graph holds, what runs between its replays
SMALL = {"run": (run("trt", 6), run("trt", 10)), "single steps": (two_steps, run("trt", 6)),
         "f32s": (run("bgk", 4), run("bgk", 6)), "op": (op(6), op(4)),
         "step and op": (two_steps, op(6)), "dugks": (dugks, dugks),
         "single dugks": (dugks, two_dugks_steps), "run and dugks": (run("trt", 6), dugks)}


@pytest.mark.parametrize("kind", list(SMALL))
def test_small_grids(P, gpu, kind):
    print(f"case graph {kind}", flush=True)
    storage = "f32s" if kind == "f32s" else "f64"
    lat, ref = lattice(P, 96, 80, storage), lattice(P, 96, 80, storage)
    single_steps(ref, storage)
    replay_between_runs(lat, ref, *SMALL[kind], both_slots(lat, ref))


@pytest.mark.parametrize("steps", [16, 32])
@pytest.mark.parametrize("nx,ny", [(600, 500), (700, 640)])
def test_medium_grids(P, gpu, nx, ny, steps):
    """Grids that take tiles and gave the column walk 512 wavefronts."""
    print(f"case graph run {nx}x{ny} {steps} steps", flush=True)
    lat, ref = lattice(P, nx, ny), lattice(P, nx, ny)
    single_steps(ref)
    replay_between_runs(lat, ref, run("trt", steps), run("trt", steps), latest_slot(lat, ref))


def test_large_operator_grid(P, gpu):
    """At least 2048 walks of 64 columns: passes of 3, four of them."""
    print("case graph op 43712x120", flush=True)
    lat, ref = lattice(P, 43712, 120), lattice(P, 43712, 120)
    single_steps(ref)
    replay_between_runs(lat, ref, op(12), op(12), latest_slot(lat, ref))
