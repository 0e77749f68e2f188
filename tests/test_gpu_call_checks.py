"""The array checks of evaluate_ and evaluate_adjoint_: arrays with the plan's
own layouts skip the property-by-property checks, so every array that fails
one of those must still be refused, with the same error, and every array that
fits in another layout must still be taken -- before and after a plan exists.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import make_dims

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[False, True], ids=["no_plan", "plan"])
def grid(gpu, request):
    g = gpu.NURBSGrid(tuple(make_dims(gpu, (7, 5), (3, 2), (19, 1))), 2)
    if request.param:
        gpu.evaluate_(g)
    return g


@pytest.mark.parametrize("adjoint", [False, True], ids=["forward", "adjoint"])
def test_refusals(gpu, grid, adjoint):
    sg = gpu
    if adjoint:
        grid = sg.SplineGrid(grid.spline_dimensions, 2)
    run = sg.evaluate_adjoint_ if adjoint else sg.evaluate_
    cp = sg.colmajor_zeros((7, 5, 2), torch.float32, "cuda")
    ev = sg.colmajor_zeros((19, 1, 2), torch.float32, "cuda")
    with pytest.raises(AssertionError, match="size\\(control_points\\)"):
        run(grid, control_points=cp[:6])
    with pytest.raises(AssertionError, match="size\\(eval\\)"):
        run(grid, eval=ev[:18])
    with pytest.raises(TypeError, match="eval has value type"):
        run(grid, eval=ev.double())
    with pytest.raises(ValueError, match="on cpu"):
        run(grid, eval=ev.cpu())
    with pytest.raises(ValueError, match="column-major"):
        run(grid, control_points=torch.zeros(7, 5, 2, device="cuda"))
    with pytest.raises(ValueError, match="Invalid derivative order"):
        run(sg.SplineGrid(grid.spline_dimensions, 2), derivative_order=(1, 0))
    with pytest.raises(AssertionError, match="one entry per input dimension"):
        run(sg.SplineGrid(grid.spline_dimensions, 2), derivative_order=(0,))
    with pytest.raises(KeyError):
        run(grid, tier="fp8")
    run(grid, control_points=cp, eval=ev)


def test_other_layouts_of_the_same_array(gpu, grid):
    """A dimension of one sample may have any stride."""
    sg = gpu
    rng = np.random.default_rng(0)
    grid.control_points.copy_(rng.uniform(-1, 1, (7, 5, 2)).astype(np.float32))
    sg.evaluate_(grid)
    odd = torch.empty_strided((19, 1, 2), (1, 977, 19), device="cuda")
    sg.evaluate_(grid, eval=odd)
    assert torch.equal(odd, grid.eval)


def test_replaced_control_points(gpu, grid):
    """Arrays are compared with the grid's current arrays, not the plan's."""
    sg = gpu
    sg.evaluate_(grid)
    grid.control_points = sg.DefaultControlPoints(
        sg.colmajor_zeros((6, 5, 2), torch.float32, "cuda"))
    with pytest.raises(AssertionError, match="size\\(control_points\\)"):
        sg.evaluate_(grid, control_points=sg.colmajor_zeros((7, 5, 2), torch.float32, "cuda"))


def test_spline_eval_backward_writes_every_entry(gpu):
    """The gradient is written, not accumulated: control points that no sample
    reaches get 0 whatever the memory held."""
    sg = gpu
    t = np.linspace(0.0, 0.2, 30)
    dims = make_dims(sg, (40, 6), (2, 2), (30, 11), sample_points=[t, None])
    for nurbs in (False, True):
        g = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(dims), 1)
        P = torch.rand(40, 6, 1, device="cuda", requires_grad=True)
        junk = torch.full((40 * 6,), float("nan"), device="cuda")
        del junk
        grad, = torch.autograd.grad(sg.spline_eval(g, P).sum(), P)
        assert bool((grad[:9] > 0).all()) and bool((grad[11:] == 0).all())
