"""The adjoint with Inf or NaN among the cotangents, the weights or the 1 / w(x):
each reaches the control points whose bands hold it, in every dimension, and
no other one, on the matrix cores as in the sums of the oracle; the finite
rest is as accurate as ever.  The shapes are tiles of 64 and 32 samples,
workgroups of four, two and one waves, 2-D and 3-D, with partial tiles.  The
bars are the repository's: 1e-6 (FP32), 1e-12 (FP64) of the largest finite
value, and 1e-5 for the FP32 NURBS adjoint.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from helpers import eval_host, make_dims, oracle_dims, rel_err

pytestmark = pytest.mark.gpu

CASES = [  # (n, p, m, nout)
    ((30, 26, 19), (3, 3, 3), (131, 150, 90), 3),
    ((40, 20, 8), (3, 3, 4), (150, 100, 21), 2),   # tiles of 32 samples
    ((9, 30, 12), (2, 3, 2), (67, 64, 33), 4),     # two waves per workgroup
    ((12, 20, 9), (3, 3, 1), (129, 31, 17), 1),    # one wave per workgroup
    ((70, 30), (3, 3), (2048, 1101), 2),           # several row blocks per wave
    ((26, 10), (2, 3), (131, 200), 4),
    ((12, 6, 5), (3, 2, 2), (65, 20, 9), 1),       # a tile of one sample
]


def _plant(a, rng, count):
    """Inf, -Inf and NaN at random places and at the ends of rows and tiles."""
    m = a.shape
    spots = [tuple(int(rng.integers(0, k)) for k in m) for _ in range(count)]
    spots.append((m[0] - 1,) + tuple(k // 2 for k in m[1:]))
    spots.append((0, m[1] // 3) + tuple(k // 3 for k in m[2:]))
    spots.append((min(63, m[0] - 1), m[1] // 2) + tuple(k // 4 for k in m[2:]))
    for i, at in enumerate(spots):
        a[at] = [np.inf, np.nan, -np.inf][i % 3]


def _check(got, want, bar):
    finite = np.isfinite(want)
    assert finite.any() and not finite.all()
    assert np.array_equal(np.isfinite(got), finite)
    assert rel_err(got[finite], want[finite]) < bar


@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("what", ["bspline", "nurbs", "weights", "zero_w"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"n{c[0]}m{c[2]}c{c[3]}")
def test_nonfinite_values_stay_in_their_bands(gpu, case, what, dtype):
    sg = gpu
    n, p, m, nout = case
    dims = make_dims(sg, n, p, m, dtype=dtype)
    nurbs = what != "bspline"
    grid = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(dims), nout)
    assert "adjoint=mma_f32+mma_f64" in grid.plan().describe()
    rng = np.random.default_rng(sum(m) + nout)
    E = rng.standard_normal(tuple(m) + (nout,)).astype(dtype)
    W = rng.uniform(0.5, 2.0, n).astype(dtype)
    if what == "weights":
        W[tuple(k // 2 for k in n)] = np.inf
        W[(n[0] - 1,) + (0,) * (len(n) - 1)] = np.nan
    elif what == "zero_w":  # w(x) = 0 at the first sample of every dimension
        W[(0,) * len(n)] = 0.0
    else:
        _plant(E, rng, 2)
    if nurbs:
        grid.weights.copy_(sg.from_numpy_colmajor(W, grid.dtype, "cuda"))
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    Pbar = sg.colmajor_zeros(tuple(n) + (nout,), grid.dtype, "cuda")
    run = sg.evaluate_rational_adjoint_ if nurbs else sg.evaluate_adjoint_
    E64, W64 = E.astype(np.float64), W.astype(np.float64)
    with np.errstate(all="ignore"):
        want = (O.adjoint_rational(oracle_dims(dims), W64, E64, nthreads=8) if nurbs
                else O.adjoint_direct(oracle_dims(dims), E64, nthreads=8))
    bar = 1e-12 if dtype == np.float64 else 1e-5 if nurbs else 1e-6
    run(grid, eval=ebar, control_points=Pbar)
    _check(eval_host(sg, Pbar), want, bar)


@pytest.mark.parametrize("how", ["f32", "f64", "nurbs_f32", "nurbs_f64", "split_f16", "bf16"])
def test_row_end_is_not_the_next_row(gpu, how):
    """The last tile's loads cross the end of a row: an Inf at the start of the
    next row does not reach the control points that only the last tile holds.
    (The tiers, which do not go back over such values, fail without the mask.)"""
    sg = gpu
    n, p, m = (28, 6, 5), (3, 2, 2), (85, 20, 9)  # tiles of 32 samples, the last of 21
    dtype = np.float64 if how.endswith("f64") else np.float32
    dims = make_dims(sg, n, p, m, dtype=dtype)
    nurbs = how.startswith("nurbs")
    grid = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(dims), 1)
    assert "adjm=32x" in grid.plan().describe(), grid.plan().describe()
    E = np.random.default_rng(5).standard_normal(m + (1,)).astype(dtype)
    E[0, 7, 4, 0] = np.inf
    ebar = sg.from_numpy_colmajor(E, grid.dtype, "cuda")
    Pbar = sg.colmajor_zeros(n + (1,), grid.dtype, "cuda")
    if nurbs:
        sg.evaluate_rational_adjoint_(grid, eval=ebar, control_points=Pbar)
    else:
        sg.evaluate_adjoint_(grid, eval=ebar, control_points=Pbar,
                             tier=how if how in ("split_f16", "bf16") else "native")
    got = eval_host(sg, Pbar)
    spans = grid.spline_dimensions[0].sample_indices.cpu().numpy() - 1  # last control point
    own = got[int(spans[63]) + 1:]  # past what the tiles before the last reach
    assert own.size > 0 and spans[63] > spans[31]
    assert not np.isfinite(got).all() and np.isfinite(own).all()
