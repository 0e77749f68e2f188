"""A batch's queues at their corners: fewer grids than XCDs (empty queues),
queues of very different lengths (workgroups past a queue's end), and the row
counts that few tiles choose, against each grid's own evaluation.  The bars
are the batch tests': 1e-6 of max|eval| natively, bit-identical for the
MFMA tiers.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import make_dims

pytestmark = pytest.mark.gpu

SPECS = [  # (n, p, m, nout, nurbs)
    ((20, 18), (3, 2), (300, 280), 3, True),
    ((12, 9, 8), (2, 3, 1), (70, 33, 21), 1, False),
    ((9, 7), (1, 4), (5, 3), 4, False),
    ((16, 16, 16), (3, 3, 3), (130, 65, 30), 3, True),
]


@pytest.mark.parametrize("count", [1, 3, 9, 30])
@pytest.mark.parametrize("tier", ["native", "split_f16"])
def test_batch_queue_corners(gpu, count, tier):
    sg = gpu
    rng = np.random.default_rng(count)
    grids = []
    for i in range(count):
        n, p, m, nout, nurbs = SPECS[i % len(SPECS)] if i else SPECS[3]
        g = (sg.NURBSGrid if nurbs else sg.SplineGrid)(tuple(make_dims(sg, n, p, m)), nout)
        g.control_points.copy_(rng.uniform(-1, 1, n + (nout,)).astype(np.float32))
        if nurbs:
            g.weights.copy_(sg.from_numpy_colmajor(
                rng.uniform(0.5, 2, n).astype(np.float32), g.dtype, "cuda"))
        grids.append(g)
    batch = sg.SplineGridBatch(grids)
    for g in grids:
        g.eval.fill_(float("nan"))
    batch.evaluate_(tier=tier)
    got = [g.eval.clone() for g in grids]
    for g, value in zip(grids, got):
        sg.evaluate_(g, tier=tier)
        if tier == "native":
            assert float((g.eval - value).abs().max()) <= 1e-6 * float(g.eval.abs().max())
        else:
            assert torch.equal(g.eval, value)
