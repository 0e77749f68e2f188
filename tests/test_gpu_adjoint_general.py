"""The general adjoint (any Nin, degree and sample order) against the oracle,
at the sizes where its threads per control point change and where a thread's,
wave's or workgroup's last pass over a band list is partial or empty.

The bar is the summation bound: a control point sums its K entries as at most
d = K / G + log2 G + G / 64 + 2 additions deep (G >= 1 threads), each entry
Nin + 1 roundings, so |error| <= (d + Nin + 2) u sum|B e|, with u the unit
roundoff; the oracle run on |e| gives sum|B e| where every B is >= 0.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import eval_host, make_dims, oracle_dims

pytestmark = pytest.mark.gpu

# (n, p, m, nout, unsorted samples)
CASES = [
    ((5,), (3,), (1,), 1, False),            # most control points without a sample
    ((30,), (3,), (360,), 2, False),         # 48 entries: one thread each
    ((30,), (3,), (370,), 2, False),         # just past it: a wave each
    ((10,), (4,), (2048,), 3, False),        # 1024 entries: the last wave case
    ((10,), (3,), (2600,), 1, False),        # 1040 entries: a workgroup each
    ((7,), (0,), (30011,), 2, False),        # degree 0, several passes
    ((40, 11), (6, 2), (90, 77), 2, False),  # degree > 5: a wave each
    ((6, 5), (3, 2), (130, 111), 1, True),   # unsorted samples, a workgroup each
    ((4, 3, 5, 4), (2, 1, 2, 3), (9, 8, 7, 6), 3, False),  # four dimensions
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{c[0]}m{c[2]}")
def test_general_adjoint_vs_oracle(gpu, case, dtype):
    sg = gpu
    n, p, m, nout, unsorted = case
    rng = np.random.default_rng(sum(m) + nout)
    points = [rng.permutation(np.linspace(0, 1, k)) for k in m] if unsorted else None
    dims = make_dims(sg, n, p, m, dtype=dtype, sample_points=points)
    grid = sg.SplineGrid(tuple(dims), nout)
    E = rng.standard_normal(tuple(m) + (nout,)).astype(dtype)
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    base = rng.standard_normal(tuple(n) + (nout,)).astype(dtype)
    Pbar = sg.from_numpy_colmajor(base, grid.dtype, "cuda")
    odims = oracle_dims(dims)
    want = O.adjoint_direct(odims, E.astype(np.float64), nthreads=8)
    size = O.adjoint_direct(odims, np.abs(E).astype(np.float64), nthreads=8)
    entries = max(np.prod([np.count_nonzero(d.dense(), axis=0).max() for d in odims]), 1)
    u = np.finfo(dtype).eps / 2
    bar = (entries + 16 + 2 + len(n) + 2) * u * size + u * np.abs(base) + 1e-300
    # a list of up to 64 * 64 entries is at least 48 entries or one thread's
    # own sum; longer ones are split over at least 64 threads
    if entries > 48 * 4:
        bar = (entries / 64 + 16 + 16 + len(n) + 4) * u * size + u * np.abs(base) + 1e-300
    sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar)
    first = eval_host(sg, Pbar)
    assert np.all(np.abs(first - want) <= bar), np.max(np.abs(first - want) / bar)
    sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar)
    assert np.array_equal(eval_host(sg, Pbar), first)  # overwritten, bit for bit
    Pbar.copy_(sg.from_numpy_colmajor(base, grid.dtype, "cuda"))
    sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar, accumulate=True)
    total = eval_host(sg, Pbar)
    assert np.all(np.abs(total - (want + base)) <= bar + u * np.abs(total))
