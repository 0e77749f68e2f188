"""Forward tiles on both sides of each line of their rule: whole and split
64-byte sectors, 4 to 32 bytes per sample, rows that one, two or four waves
fill, 2-D and 3-D, few and many workgroups, last tiles and chunks that are not
full.  Values against the oracle at the repository's bars (1e-6 and 1e-12 of
max|oracle|); the expected tile is width x rows of a workgroup.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import (TOL, clamped_knot_vector, eval_host, make_dims, oracle_dims,
                     random_cp, rel_err)

pytestmark = pytest.mark.gpu

CASES = [  # n, p, m, nout, tile FP32, tile FP64
    ((4, 5, 4), (1, 2, 2), (1, 7, 5), 1, "64x32", "64x32"),
    ((9, 8, 6), (2, 3, 1), (45, 33, 30), 2, "64x32", "64x32"),
    ((9, 8, 6), (3, 2, 3), (64, 40, 10), 2, "64x32", "64x32"),
    ((30, 12, 8), (2, 2, 2), (300, 100, 40), 4, "64x32", "64x32"),
    ((30, 15, 14), (2, 2, 2), (300, 150, 140), 4, "64x32", "64x32"),
    ((20, 14, 12), (3, 3, 3), (203, 130, 110), 1, "256x32", "256x16"),
    ((16, 9, 12), (3, 1, 2), (130, 65, 90), 3, "64x64", "64x64"),
    ((13, 9, 20), (2, 3, 2), (127, 70, 200), 3, "128x32", "128x32"),
    ((60, 70), (3, 3), (1501, 1700), 3, "256x16", "256x16"),
    ((40, 30), (2, 4), (1032, 900), 2, "128x16", "128x16"),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("nurbs", [False, True], ids=["bspline", "nurbs"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"m{c[2]}c{c[3]}")
def test_forward_tiles_vs_oracle(gpu, case, nurbs, dtype):
    sg = gpu
    n, p, m, nout, tile32, tile64 = case
    rng = np.random.default_rng(sum(m) + nout)
    dims = make_dims(sg, n, p, m, dtype=dtype)
    grid = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(dims), nout)
    P = random_cp(rng, n, nout, dtype)
    W = rng.uniform(0.5, 2.0, n).astype(dtype) if nurbs else None
    grid.control_points.copy_(sg.from_numpy_colmajor(P, grid.dtype, "cuda"))
    if nurbs:
        grid.weights.copy_(sg.from_numpy_colmajor(W, grid.dtype, "cuda"))
    desc = grid.plan().describe()
    assert f"fwd={tile32}x1," in desc and f"fwd_f64={tile64}x1," in desc, desc
    grid.eval.fill_(float("nan"))
    sg.evaluate_(grid)
    want = O.eval_direct(oracle_dims(dims), P.astype(np.float64),
                         W=W.astype(np.float64) if nurbs else None)
    assert rel_err(eval_host(sg, grid.eval), want) <= TOL[dtype]


SWEPT = [  # n, p, m: scalar volumes of 1.5 M samples and more
    ((60, 9, 30), (1, 2, 1), (517, 33, 90)),     # row tails of 1 sample; the last run is short
    ((9, 30, 40), (4, 1, 4), (38, 203, 201)),    # many rows per tile, last tile not full
    ((170, 8, 12), (3, 3, 2), (2051, 19, 40)),   # several tiles per row
    ((4, 200, 24), (2, 4, 3), (3, 2100, 260)),   # rows shorter than one store
    ((64, 40, 48), (3, 3, 3), (256, 128, 128)),  # whole tiles
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("case", SWEPT, ids=lambda c: f"m{c[2]}p{c[1]}")
def test_swept_volume_vs_oracle(gpu, case, dtype):
    """Scalar volumes on the swept kernel, value and mixed derivative; knot
    lines doubled in dimension 3, so that a span advances by two."""
    sg = gpu
    n, p, m = case
    rng = np.random.default_rng(sum(m))
    kv3 = clamped_knot_vector(sg, np.linspace(0, 1, n[2] - p[2] - 1 + 2 * (p[2] < 2)), p[2], dtype,
                              doubled=(2, 3) if p[2] > 1 else ())
    dims = make_dims(sg, n, p, m, D=[1, 1, 1], dtype=dtype, knot_vectors=[None, None, kv3])
    grid = sg.SplineGrid(tuple(dims), 1)
    P = random_cp(rng, n, 1, dtype)
    grid.control_points.copy_(sg.from_numpy_colmajor(P, grid.dtype, "cuda"))
    assert "forward=sweep" in grid.plan().describe(), grid.plan().describe()
    for orders in ((0, 0, 0), (1, 0, 1)):
        grid.eval.fill_(float("nan"))
        sg.evaluate_(grid, derivative_order=orders)
        want = O.eval_direct(oracle_dims(dims), P.astype(np.float64), deriv=orders)
        assert rel_err(eval_host(sg, grid.eval), want) <= TOL[dtype]


def test_small_and_many_channel_volumes_stream(gpu):
    sg = gpu
    for n, m, nout in (((9, 9, 9), (64, 64, 64), 1), ((40, 30, 20), (200, 100, 90), 2),
                       ((100, 100, 90), (120, 120, 110), 1)):
        grid = sg.SplineGrid(tuple(make_dims(sg, n, (2, 3, 2), m)), nout)
        assert "forward=stream" in grid.plan().describe(), grid.plan().describe()
