"""The general adjoint with one thread per control point, against the oracle:
two to eight dimensions, lists that are empty, and the many outputs of longer
lists that keep a thread each.

The bar is the summation bound: K entries in a row, each Nin + 1 roundings, so
|error| <= (K + Nin + 2) u sum|B e|, with u the unit roundoff; the oracle run
on |e| gives sum|B e| (every B is >= 0).
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import eval_host, make_dims, oracle_dims

pytestmark = pytest.mark.gpu

# (n, p, m, nout, unsorted samples)
CASES = [
    ((9, 7), (6, 1), (13, 5), 3, False),
    ((40, 9), (6, 2), (11, 9), 1, False),       # control points without a sample
    ((300, 300), (6, 6), (350, 350), 2, False),  # 67 entries, 180 000 outputs
    ((8, 9, 8), (6, 2, 1), (9, 11, 7), 2, False),
    ((6, 5, 7), (1, 2, 1), (9, 11, 7), 1, True),
    ((4, 3, 5, 4), (1, 1, 2, 1), (5, 3, 6, 4), 3, False),
    ((3, 2, 3, 2, 3), (1, 1, 1, 1, 1), (3, 2, 4, 2, 3), 2, True),
    ((2,) * 6, (1,) * 6, (2, 3, 2, 1, 2, 2), 1, False),
    ((2,) * 7, (1,) * 7, (2, 1, 2, 1, 2, 2, 1), 1, False),
    ((2,) * 8, (1,) * 8, (1, 2, 1, 2, 1, 1, 2, 2), 2, False),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{c[0]}m{c[2]}")
def test_thread_per_control_point_vs_oracle(gpu, case, dtype):
    sg = gpu
    n, p, m, nout, unsorted = case
    rng = np.random.default_rng(sum(m) + nout)
    points = [rng.permutation(np.linspace(0, 1, k)) for k in m] if unsorted else None
    dims = make_dims(sg, n, p, m, dtype=dtype, sample_points=points)
    grid = sg.SplineGrid(tuple(dims), nout)
    E = rng.standard_normal(tuple(m) + (nout,)).astype(dtype)
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    Pbar = sg.from_numpy_colmajor(np.full(tuple(n) + (nout,), np.nan, dtype), grid.dtype, "cuda")
    odims = oracle_dims(dims)
    want = O.adjoint_direct(odims, E.astype(np.float64), nthreads=8)
    size = O.adjoint_direct(odims, np.abs(E).astype(np.float64), nthreads=8)
    entries = np.prod([np.count_nonzero(d.dense(), axis=0).max() for d in odims])
    u = np.finfo(dtype).eps / 2
    bar = (entries + len(n) + 2) * u * size + 1e-300
    sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar)
    got = eval_host(sg, Pbar)
    assert np.all(np.abs(got - want) <= bar), np.max(np.abs(got - want) / bar)
    sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar, accumulate=True)
    total = eval_host(sg, Pbar)
    assert np.all(np.abs(total - 2 * want) <= 2 * bar + u * np.abs(total))
