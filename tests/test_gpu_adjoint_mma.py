"""The matrix-core adjoint, FP32 and FP64, B-spline and NURBS, against the
oracle where its tiles are partial: rows shorter than one 16-byte load, rows
whose last load crosses the row's end, tiles of 32 samples, workgroups of one,
two and four waves with waves that have no rows, 2-D grids with several row
blocks per wave, runs of j3 that end inside a knot span, and channel groups
that are not full.  The bars are the repository's: 1e-6 (FP32), 1e-12 (FP64)
of max|oracle|, and 1e-5 for the FP32 NURBS adjoint.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import eval_host, make_dims, oracle_dims, rel_err

pytestmark = pytest.mark.gpu

CASES = [
    ((4, 5, 4), (1, 2, 2), (1, 9, 5), 1),
    ((4, 5, 4), (1, 2, 3), (2, 18, 7), 4),
    ((5, 4), (2, 1), (3, 65), 2),
    ((7, 9, 5), (3, 3, 1), (63, 61, 9), 2),
    ((9, 8, 6), (3, 2, 3), (65, 17, 40), 3),
    ((9, 30, 12), (2, 3, 2), (67, 64, 33), 5),     # two waves per workgroup
    ((12, 20, 9), (3, 3, 0), (129, 31, 17), 1),    # one wave per workgroup
    ((40, 20, 8), (3, 3, 4), (150, 100, 21), 2),   # tiles of 32 samples
    ((30, 12, 9), (4, 2, 5), (97, 100, 60), 3),    # tiles of 32 samples, p3 = 5
    ((70, 30), (3, 3), (2048, 1101), 2),           # 2-D, several row blocks per wave
    ((26, 10), (2, 3), (131, 200), 4),             # 2-D, one row block per wave
]


def _inputs(sg, case, dtype, nurbs):
    n, p, m, nout = case
    dims = make_dims(sg, n, p, m, dtype=dtype)
    grid = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(dims), nout)
    rng = np.random.default_rng(sum(m) + 7 * nout)
    E = rng.standard_normal(tuple(m) + (nout,)).astype(dtype)
    W = rng.uniform(0.5, 2.0, n).astype(dtype)
    if nurbs:
        grid.weights.copy_(sg.from_numpy_colmajor(W, grid.dtype, "cuda"))
    assert "adjoint=mma_f32+mma_f64" in grid.plan().describe(), grid.plan().describe()
    return dims, grid, E, W


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("nurbs", [False, True], ids=["bspline", "nurbs"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{c[0]}m{c[2]}c{c[3]}")
def test_adjoint_mma_vs_oracle(gpu, case, nurbs, dtype):
    sg = gpu
    dims, grid, E, W = _inputs(sg, case, dtype, nurbs)
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    Pbar = sg.colmajor_zeros(tuple(case[0]) + (case[3],), grid.dtype, "cuda")
    run = sg.evaluate_rational_adjoint_ if nurbs else sg.evaluate_adjoint_
    E64 = E.astype(np.float64)
    want = (O.adjoint_rational(oracle_dims(dims), W.astype(np.float64), E64, nthreads=8) if nurbs
            else O.adjoint_direct(oracle_dims(dims), E64, nthreads=8))
    bar = 1e-12 if dtype == np.float64 else 1e-5 if nurbs else 1e-6
    run(grid, eval=ebar, control_points=Pbar)
    first = eval_host(sg, Pbar)
    assert rel_err(first, want) < bar
    run(grid, eval=ebar, control_points=Pbar, accumulate=True)
    assert rel_err(eval_host(sg, Pbar), 2 * want) < bar
    run(grid, eval=ebar, control_points=Pbar)
    assert np.array_equal(eval_host(sg, Pbar), first)


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("nurbs", [False, True], ids=["bspline", "nurbs"])
def test_row_end_does_not_read_the_next_row(gpu, nurbs, dtype):
    """An infinite sample at the start of a row stays out of the control points
    that only the end of the row before it reaches."""
    sg = gpu
    case = ((12, 6, 5), (3, 2, 2), (65, 20, 9), 1)
    _, grid, E, _ = _inputs(sg, case, dtype, nurbs)
    E[0, 7, 4, 0] = np.inf
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    Pbar = sg.colmajor_zeros(tuple(case[0]) + (case[3],), grid.dtype, "cuda")
    run = sg.evaluate_rational_adjoint_ if nurbs else sg.evaluate_adjoint_
    run(grid, eval=ebar, control_points=Pbar)
    got = eval_host(sg, Pbar)
    # tile 1 (sample 64 alone) reaches the last four control points; the last
    # one has no sample of tile 0 but 63 and below whose B there is not 0
    assert np.isinf(got[0]).any() or np.isnan(got[0]).any()
    first_tile = int(grid.spline_dimensions[0].sample_indices[63]) - 1  # last span of tile 0
    assert np.isfinite(got[first_tile + 1:]).all()
