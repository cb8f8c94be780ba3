"""Batches of long cases of few columns, which walk, and of others, some of them such, which run in
tiles: every case against a single lattice of its own in single steps, FP64, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BATCHES = {"slender": [(4, 1600), (1, 2003), (7, 2900), (3, 5)],
           "slender with one other": [(4, 1700), (2, 1500), (40, 30)],
           "mixed": [(4, 1600), (64, 70), (8, 3200), (33, 64)]}


@pytest.mark.parametrize("sizes", [[(4, 2000)] * 40, [(1, 400), (7, 2800), (7, 100)]])
def test_slender_cases_walk(P, gpu, sizes):
    """As with the walk's columns set, to the rounding of FP32 collisions (whose FMAs tiles place
    otherwise)."""
    rng = np.random.default_rng(6)
    fields = [[m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)]
              for nx, ny in sizes]
    out = []
    for columns in (None, 64):
        b = P.Batch(sizes, "f32s", "trt")
        b.set_params([1.7] * len(sizes), [0.25] * len(sizes))
        b.set_steps_per_pass(6)
        if columns:
            b.set_pass_columns(columns)
        for c, m in enumerate(fields):
            b.equilibrium_init(c, *m)
        b.run(40)
        out.append([b.download_f(c) for c in range(len(sizes))])
    for a, w in zip(*out):
        np.testing.assert_array_equal(a, w)


@pytest.mark.parametrize("per_pass", [2, 6, 8])
@pytest.mark.parametrize("model", ["bgk", "trt"])
@pytest.mark.parametrize("kind", list(BATCHES))
def test_cases(P, gpu, kind, model, per_pass):
    print(f"case batch {kind} {model} passes of {per_pass}", flush=True)
    sizes, rng = BATCHES[kind], np.random.default_rng(5)
    b = P.Batch(sizes, "f64", model)
    b.set_params([1.7] * len(sizes), [0.25] * len(sizes))
    b.set_steps_per_pass(per_pass)
    fields = [[m + 0.02 * rng.standard_normal((ny, nx)) for m in (1.0, 0.0, 0.0)]
              for nx, ny in sizes]
    for c, m in enumerate(fields):
        b.equilibrium_init(c, *m)
    b.run(19)
    for c, (nx, ny) in enumerate(sizes):
        lat = P.Lattice(nx, ny, 2, "f64")
        lat.set_params(1.7, 0.25)
        lat.set_steps_per_launch(model, 1)
        lat.equilibrium_init(0, *fields[c])
        i, _ = lat.run(model, 19, 0, 1)
        np.testing.assert_array_equal(b.download_f(c)[:ny], lat.download_f(i)[:ny])
