"""The adjoint of a long thin volume: more (k3, channel) planes of a few control
points than one launch of the gather holds.

With ebar[j, c] = (c + 1) f(j3) the adjoint is the product of the dimensions'
column sums, (c + 1) s1[k1] s2[k2] (B3^T f)[k3], formed here in FP64; every
term is positive and a control point sums at most 36 of them, so the bar is
(36 + 8) u of the value, u the unit roundoff of FP32.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import make_dims

pytestmark = pytest.mark.gpu


def test_more_planes_than_a_launch(gpu):
    sg = gpu
    n3, nout = (1 << 22) + 3, 4  # planes of 256 threads: over 2^32 threads
    n, m = (2, 2, n3), (3, 3, n3)
    dims = make_dims(sg, n, (1, 1, 1), m)
    out = sg.colmajor_empty(m + (nout,), torch.float32, "cuda")
    grid = sg.SplineGrid(tuple(dims), sg.colmajor_zeros(n + (nout,), torch.float32, "cuda"), None,
                         out)
    assert "adjoint=mma_f32" in grid.plan().describe()
    f = 1.0 + (torch.arange(n3, device="cuda") % 7)
    c = 1.0 + torch.arange(nout, device="cuda")
    out.copy_((f[:, None] * c[None, :])[None, None])
    got = sg.colmajor_empty(n + (nout,), torch.float32, "cuda").fill_(float("nan"))
    sg.evaluate_adjoint_(grid, eval=out, control_points=got)

    def columns(s, weight):  # sum_j B[j, k] weight[j]
        first = s.sample_indices.long() - s.degree - 1
        total = torch.zeros(s.n_basis_functions, dtype=torch.float64, device="cuda")
        for a in range(s.degree + 1):
            total.index_add_(0, first + a, s.eval[:, a, 0].double() * weight)
        return total

    ones = torch.ones(3, dtype=torch.float64, device="cuda")
    s1, s2, s3 = columns(dims[0], ones), columns(dims[1], ones), columns(dims[2], f.double())
    u = float(np.finfo(np.float32).eps) / 2
    for ch in range(nout):
        want = (ch + 1) * s1[:, None, None] * s2[None, :, None] * s3[None, None, :]
        assert bool(((got[..., ch].double() - want).abs() <= (36 + 8) * u * want).all())
