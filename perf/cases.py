"""Workloads of the grid-evaluation framework for timing.

A case is one call (or one forward + backward) on a grid as a program keeps
it: dimensions with default clamped knots and uniform samples, control
points, weights and an output array on the GPU.  ``kind`` says which public
entry point a pass goes through:

  forward           evaluate_(grid)                      curve / surface / volume evaluation
  fields            evaluate_fields_(grid, orders)       value and partial derivatives at once
  adjoint           evaluate_adjoint_(grid)              gradient of a loss in the control points
  train             spline_eval + its backward           one differentiable evaluation
  nurbs_fields      evaluate_rational_fields_            derivatives of a NURBS map
  nurbs_adjoint     evaluate_rational_adjoint_           gradient through a NURBS map
  batch             SplineGridBatch.evaluate_            many uneven grids in one call

n, p and m are control points, degree and samples per dimension, written as
text ("64x64x32") so that a case holds plain values only.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import __graft_entry__

DEVICE = "cuda"

# requested derivative orders of the "fields" kinds, by input dimensions
FIELDS = {2: [(0, 0), (1, 0), (0, 1), (1, 1)],
          3: [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]}
GRADIENT = {2: [(1, 0), (0, 1)], 3: [(1, 0, 0), (0, 1, 0), (0, 0, 1)]}


def _case(kind, n, p, m, nout, dtype="f32", nurbs=False, tier="native", name=None):
    c = dict(kind=kind, n="x".join(map(str, n)), p="x".join(map(str, p)),
             m="x".join(map(str, m)), nout=nout, dtype=dtype, nurbs=nurbs, tier=tier)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a surface patch re-evaluated inside a loop: nothing but latency
        _case("forward", (10, 12), (2, 3), (25, 31), 3, nurbs=True, name="patch_nurbs_f32"),
        # the volume of the README, in the precision that fits are run in
        _case("forward", (10, 10, 5), (2, 3, 2), (50, 50, 25), 4, dtype="f64",
              name="readme_volume_f64"),
        # a curve through many measured points, one step of its fit
        _case("train", (101,), (3,), (20011,), 2, name="curve_train_f32"),
        # an image-sized surface of odd sides, one step of its fit
        _case("train", (61, 47), (3, 3), (1027, 773), 3, name="surface_train_f32"),
        # a deformation field over a volume of odd sides, one step of its fit
        _case("train", (33, 29, 17), (3, 3, 3), (251, 197, 123), 3,
              name="volume_train_ragged_f32"),
        # gradient of a loss over a large volume
        _case("adjoint", (40, 40, 20), (3, 3, 3), (400, 400, 200), 3, name="volume_adjoint_f32"),
        # the same in double precision, as a least-squares fit runs it
        _case("adjoint", (40, 40, 20), (3, 3, 3), (200, 201, 99), 3, dtype="f64",
              name="volume_adjoint_f64"),
        # a fine surface with its derivatives (normals, metric)
        _case("fields", (128, 128), (3, 3), (4096, 4096), 1, name="surface_fields_f32"),
        # a large NURBS volume: evaluation, its derivatives, its adjoint
        _case("forward", (64, 64, 32), (3, 3, 2), (512, 512, 256), 3, nurbs=True,
              name="nurbs_volume_f32"),
        _case("nurbs_fields", (64, 64, 32), (3, 3, 2), (512, 512, 256), 3, nurbs=True,
              name="nurbs_gradient_f32"),
        _case("nurbs_adjoint", (64, 64, 32), (3, 3, 2), (512, 512, 256), 3, nurbs=True,
              name="nurbs_adjoint_f32"),
        # many patches and blocks of uneven sizes, half surfaces, half volumes
        dict(name="batch_uneven_f32", kind="batch", grids=256, spec=5, dtype="f32"),
    ]


# Sample-points a drawn case may cost at most, by kind, so that none costs
# more than the largest listed case (three fields of 67M samples x 3).
_MOST = {"forward": 6.7e7, "fields": 1.6e7, "adjoint": 3.2e7, "train": 1.6e7,
         "nurbs_fields": 4.0e7, "nurbs_adjoint": 4.0e7}


def draw(rng):
    kind = rng.choice(["forward", "forward", "fields", "adjoint", "train", "train",
                       "nurbs_fields", "nurbs_adjoint", "batch"])
    if kind == "batch":
        return dict(kind="batch", grids=round(math.exp(rng.uniform(math.log(16), math.log(256)))),
                    spec=rng.randrange(1000, 1 << 20), dtype="f32")
    lowest = 1 if kind in ("forward", "train") else 2
    nin = rng.choice([d for d in (1, 2, 2, 3, 3, 3) if d >= lowest])
    nurbs = kind.startswith("nurbs") or (kind == "forward" and rng.random() < 0.4)
    dtype = "f64" if rng.random() < 0.25 else "f32"
    tier = "native"
    if kind == "forward" and dtype == "f32" and nin >= 2 and rng.random() < 0.3:
        tier = rng.choice(["split_f16", "bf16"])
    nout = rng.choice([1, 2, 3, 3, 4])
    most = _MOST[kind] * (0.5 if dtype == "f64" else 1.0) * 3 / max(nout, 3)
    p = tuple(rng.randint(1 if kind == "forward" else 2, 4) for _ in range(nin))
    hi = {1: 2.0e5, 2: 4096.0, 3: 512.0}[nin]
    lo = {1: 100.0, 2: 24.0, 3: 16.0}[nin]
    while True:
        m = tuple(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))) for _ in range(nin))
        if math.prod(m) <= most:
            break
    # 3 to 16 samples per control point, as in fits and fine evaluations
    cap = {1: 400, 2: 160, 3: 64}[nin]
    n = tuple(max(pd + 1, min(cap, round(md / math.exp(rng.uniform(math.log(3), math.log(16))))))
              for pd, md in zip(p, m))
    return _case(kind, n, p, m, nout, dtype=dtype, nurbs=nurbs, tier=tier)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _ints(text):
    return tuple(int(x) for x in text.split("x"))


def _specs(case):
    """Every grid of a case as (n, p, m, nout, nurbs)."""
    if case["kind"] != "batch":
        return [(_ints(case["n"]), _ints(case["p"]), _ints(case["m"]), case["nout"],
                 case["nurbs"])]
    rng = np.random.default_rng(case["spec"])
    specs = []
    for i in range(case["grids"]):
        nin = 2 if i < case["grids"] // 2 else 3
        n = tuple(int(x) for x in rng.integers(8, 65, nin))
        p = tuple(int(min(rng.integers(1, 5), nd - 1)) for nd in n)
        lo, hi = (32, 513) if nin == 2 else (16, 129)
        m = tuple(int(x) for x in rng.integers(lo, hi, nin))
        specs.append((n, p, m, int(rng.choice([1, 3])), bool(rng.random() < 0.25)))
    return specs


def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _orders(case, nin):
    """Largest derivative order of each dimension's tables."""
    return [1 if case["kind"] in ("fields", "nurbs_fields") else 0] * nin


def _colmajor(flat, shape):
    return flat.view(tuple(shape)[::-1]).permute(*range(len(shape) - 1, -1, -1))


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _values(case, specs, gen):
    """(control points, weights) of every grid: P ~ U[-1, 1), W ~ U[0.5, 2)."""
    dt = _dtype(case)
    total = sum(math.prod(n) * (nout + 1) for n, _, _, nout, _ in specs)
    pool = torch.rand(total, generator=gen, dtype=dt, device=DEVICE)
    out, at = [], 0
    for n, _, _, nout, nurbs in specs:
        ncp = math.prod(n)
        P = pool[at:at + ncp * nout].mul(2).sub_(1)
        W = pool[at + ncp * nout:at + ncp * (nout + 1)].mul(1.5).add_(0.5)
        at += ncp * (nout + 1)
        out.append((_colmajor(P, n + (nout,)), _colmajor(W, n) if nurbs else None))
    return out


def _cotangent(case, spec, gen):
    _, _, m, nout, _ = spec
    flat = torch.randn(math.prod(m) * nout, generator=gen, dtype=_dtype(case), device=DEVICE)
    return _colmajor(flat, m + (nout,))


def _np_float(case):
    return np.float64 if case["dtype"] == "f64" else np.float32


def prepare(case, seed):
    sg = __graft_entry__.package()
    kind, specs, gen, dt = case["kind"], _specs(case), _generator(seed), _dtype(case)
    values = _values(case, specs, gen)
    # outputs in one allocation, each on a 256-byte boundary
    sizes = [-(-math.prod(m) * nout // 64) * 64 for _, _, m, nout, _ in specs]
    pool = torch.zeros(sum(sizes), dtype=dt, device=DEVICE)
    grids, at = [], 0
    for (n, p, m, nout, _), (P, W), size in zip(specs, values, sizes):
        dims = tuple(sg.SplineDimension(nd, pd, md, max_derivative_order=od,
                                        float_type=_np_float(case), device=DEVICE)
                     for nd, pd, md, od in zip(n, p, m, _orders(case, len(n))))
        out = _colmajor(pool[at:at + math.prod(m) * nout], m + (nout,))
        grids.append(sg.SplineGrid(dims, P, W, out))
        at += size
    state = {"sg": sg, "case": case, "grid": grids[0], "pool": pool, "grids": grids}
    if kind == "batch":
        state["batch"] = sg.SplineGridBatch(grids)
        return state
    grids[0].plan()
    nin = len(specs[0][0])
    if kind in ("adjoint", "nurbs_adjoint", "train"):
        state["cotangent"] = _cotangent(case, specs[0], gen)
    if kind in ("adjoint", "nurbs_adjoint"):
        state["gradient"] = sg.colmajor_zeros(specs[0][0] + (specs[0][3],), dt, DEVICE)
    if kind == "train":
        state["leaf"] = values[0][0].detach().requires_grad_(True)
    if kind in ("fields", "nurbs_fields"):
        orders = FIELDS[nin] if kind == "fields" else GRADIENT[nin]
        shape = specs[0][2] + (specs[0][3],)
        state["orders"] = orders
        state["fields"] = [sg.colmajor_empty(shape, dt, DEVICE) for _ in orders]
    return state


def run(state):
    sg, case, grid = state["sg"], state["case"], state["grid"]
    kind = case["kind"]
    if kind == "forward":
        sg.evaluate_(grid, tier=case["tier"])
        return grid.eval
    if kind == "fields":
        sg.evaluate_fields_(grid, state["orders"], state["fields"])
        return state["fields"]
    if kind == "adjoint":
        sg.evaluate_adjoint_(grid, eval=state["cotangent"], control_points=state["gradient"])
        return state["gradient"]
    if kind == "train":
        out = sg.spline_eval(grid, state["leaf"])
        grad, = torch.autograd.grad(out, state["leaf"], state["cotangent"])
        return out.detach(), grad
    if kind == "nurbs_fields":
        sg.evaluate_rational_fields_(grid, state["orders"], state["fields"])
        return state["fields"]
    if kind == "nurbs_adjoint":
        sg.evaluate_rational_adjoint_(grid, eval=state["cotangent"],
                                      control_points=state["gradient"])
        return state["gradient"]
    state["batch"].evaluate_()
    return state["pool"]


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

def work(case):
    """Every input read once and every output written once, and the sums of
    the banded mode products (dimension 3, then 1, then 2)."""
    size = 8 if case["dtype"] == "f64" else 4
    kind, nbytes, flops = case["kind"], 0, 0
    for n, p, m, nout, nurbs in _specs(case):
        nin, ncp, nsamp = len(n), math.prod(n), math.prod(m)
        fields = len(FIELDS[nin]) if kind == "fields" else \
            len(GRADIENT[nin]) if kind == "nurbs_fields" else 1
        passes = 2 if kind == "train" else 1
        weights = ncp if nurbs else 0
        tables = sum(md * ((pd + 1) * (od + 1) * size + 4)
                     for pd, md, od in zip(p, m, _orders(case, nin)))
        nbytes += passes * (size * (fields * nsamp * nout + ncp * nout + weights) + tables)
        sizes, sums = list(n), 0
        for d in ((2, 0, 1) if nin == 3 else range(nin)):
            sizes[d] = m[d]
            sums += math.prod(sizes) * (p[d] + 1)
        flops += 2 * sums * passes * fields * (nout + (1 if nurbs else 0))
    return {"bytes": nbytes, "flops": flops}


# --------------------------------------------------------------------------
# the same in 64 bits, with torch alone
# --------------------------------------------------------------------------

def _basis(n, p, m, order, ft):
    """Dense (m, n) matrix of the order-th derivative of the clamped uniform
    basis at uniform samples, knots and samples rounded to ft first."""
    def uniform(k):
        t = np.arange(k) / max(k - 1, 1)
        if k > 1:
            t[-1] = 1.0
        return t.astype(ft).astype(np.float64)

    values = uniform(n - p + 1)
    knots = np.concatenate([np.full(p, values[0]), values, np.full(p, values[-1])])
    t = uniform(m)
    span = np.clip(np.searchsorted(knots, t, side="right") - 1, p, n - 1)

    def local(q):
        """The q + 1 non-zero values N_{span-q..span, q}(t) (Cox-de Boor)."""
        N = np.ones((m, 1))
        for d in range(1, q + 1):
            new = np.zeros((m, d + 1))
            for a in range(d):
                k = span - d + 1 + a
                left, right = knots[k], knots[k + d]
                new[:, a] += N[:, a] * (right - t) / (right - left)
                new[:, a + 1] += N[:, a] * (t - left) / (right - left)
            N = new
        return N

    if order == 0:
        N = local(p)
    else:  # N' = p (N_{k, p-1} / (t_{k+p} - t_k) - N_{k+1, p-1} / (t_{k+p+1} - t_{k+1}))
        low, N = local(p - 1), np.zeros((m, p + 1))
        for a in range(p):
            k = span - p + 1 + a
            v = p * low[:, a] / (knots[k + p] - knots[k])
            N[:, a + 1] += v
            N[:, a] -= v
    dense = np.zeros((m, n))
    np.put_along_axis(dense, (span - p)[:, None] + np.arange(p + 1), N, axis=1)
    return torch.from_numpy(dense).to(DEVICE)


def _products(X, mats):
    """X (a_1, ..., a_d, c) with every axis d multiplied by mats[d] (b_d, a_d)."""
    for d, M in enumerate(mats):
        X = torch.movedim(torch.tensordot(M, X, dims=([1], [d])), 0, d)
    return X


def exact(case, seed):
    kind, specs, gen = case["kind"], _specs(case), _generator(seed)
    values = _values(case, specs, gen)
    ft, outs, pool = _np_float(case), [], []
    for spec, (P, W) in zip(specs, values):
        n, p, m, nout, _ = spec
        nin, P = len(n), P.double()
        W = None if W is None else W.double().unsqueeze(-1)

        def mats(order):
            return [_basis(nd, pd, md, o, ft) for nd, pd, md, o in zip(n, p, m, order)]

        zero = (0,) * nin
        if kind in ("forward", "train", "batch"):
            out = _products(P if W is None else W * P, mats(zero))
            if W is not None:
                out /= _products(W, mats(zero))
            outs.append(out)
        if kind == "batch":
            flat = outs.pop().permute(*range(nin, -1, -1)).reshape(-1)
            pool += [flat, flat.new_zeros(-flat.numel() % 64)]
        if kind == "fields":
            outs += [_products(P, mats(o)) for o in FIELDS[nin]]
        if kind == "nurbs_fields":
            w = _products(W, mats(zero))
            R = _products(W * P, mats(zero)) / w
            for o in GRADIENT[nin]:
                outs.append((_products(W * P, mats(o)) - _products(W, mats(o)) * R) / w)
        if kind in ("adjoint", "nurbs_adjoint", "train"):
            E = _cotangent(case, spec, gen).double()
            if kind == "nurbs_adjoint":
                E = E / _products(W, mats(zero))
            G = _products(E, [M.t() for M in mats(zero)])
            outs.append(W * G if kind == "nurbs_adjoint" else G)
    if kind == "batch":
        return torch.cat(pool)
    return tuple(outs) if kind == "train" else outs if "fields" in kind else outs[0]
