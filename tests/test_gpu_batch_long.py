"""A batch whose queues hold more tiles than one launch has workgroups for:
every tile of every part is evaluated.

Degree 1 with one sample in dimensions 1 and 2 is linear interpolation along
dimension 3.  Knots and samples are rounded to FP32, which moves a basis value
by at most 2 * 63 u (63 cells), and the sums round 8 times: the bar is
(126 + 8) u for control points in [0, 1), u the unit roundoff of FP32.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_queues_longer_than_a_launch(gpu):
    sg = gpu
    m3 = 4 * ((1 << 24) + 4099)  # a tile per four samples, over 2^32 threads in all
    dims = [sg.SplineDimension(2, 1, 1), sg.SplineDimension(2, 1, 1),
            sg.SplineDimension(64, 1, m3)]
    P = sg.colmajor_zeros((2, 2, 64, 1), torch.float32, "cuda")
    P.copy_(torch.from_numpy(np.random.default_rng(3).uniform(0, 1, (2, 2, 64, 1))))
    out = sg.colmajor_empty((1, 1, m3, 1), torch.float32, "cuda").fill_(float("nan"))
    batch = sg.SplineGridBatch([sg.SplineGrid(tuple(dims), P, None, out)])
    batch.evaluate_()
    x = dims[2].sample_points.double() * 63
    i = x.floor().clamp(0, 62).long()
    v = P[0, 0, :, 0].double()
    want = v[i] + (x - i) * (v[i + 1] - v[i])
    bar = (126 + 8) * float(np.finfo(np.float32).eps) / 2
    assert bool(((out[0, 0, :, 0].double() - want).abs() <= bar).all())
