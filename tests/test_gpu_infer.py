"""The fused predictor inference (hps_mlp_infer) and the difference norm.

hps_mlp_infer is compared with its own parts run one after the other
(features, layer products, correction): features, weights and the roundings
to bf16 are the same, only the FP32 accumulation order and the hidden
activations' last bits differ.  A hidden activation may therefore round to
the neighbouring bf16 value (2^-8 relative); over 128 inputs of weights of
at most 1/sqrt(128) that moves an output by far less than 2^-5 of its
hidden layer's scale, so the corrections agree to 2^-5 of their largest.
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from hpsint_amd import CartesianMesh, SinteringOperatorGeneric  # noqa: E402
from hpsint_amd._ffi import HpsError, check, lib  # noqa: E402
from hpsint_amd.predictor import MLP, LearnedPredictor  # noqa: E402


def setup(cells, G, seed=0):
    mesh = CartesianMesh(cells, (0.0,) * len(cells), tuple(float(c) for c in cells))
    op = SinteringOperatorGeneric(mesh, G)
    mlp = MLP(op, seed=seed)
    mlp.W[-1] *= 30.0
    mlp.Wb[-1].copy_(mlp.W[-1])
    for b in mlp.b:
        b.uniform_(-0.1, 0.1)
    pred = LearnedPredictor(op, mlp, dt_scale=1e3, out_scale=(0.5, 0.8, 0.4, 0.3))
    rng = np.random.default_rng(seed + 1)
    cur = torch.from_numpy(rng.uniform(0, 1, op.n_dofs)).cuda()
    prev = cur + 1e-3 * torch.from_numpy(rng.standard_normal(op.n_dofs)).cuda()
    return op, pred, prev, cur


def parts(pred, prev, cur):
    """the same prediction kernel by kernel"""
    op = pred.op
    X, top2 = pred.features(prev, cur, 1e-3)
    Y, _ = pred.mlp.forward(X, op.n_nodes)
    out = torch.empty_like(cur)
    p = ctypes.c_void_p
    check(lib().hps_mlp_predict(op.handle, p(prev.data_ptr()), p(cur.data_ptr()),
                                p(Y.data_ptr()), p(top2.data_ptr()),
                                p(pred.out_scale.data_ptr()), p(pred.lscale.data_ptr()),
                                p(out.data_ptr())))
    return out, top2.clone(), pred.lscale.clone()


# the features' tiles of 8 x 8 node columns and marches of 2 planes or more,
# the fused kernel's runs of 32 nodes
@pytest.mark.parametrize("cells,G", [
    ((1, 1, 1), 1), ((7, 7, 3), 2), ((8, 7, 1), 3), ((15, 16, 2), 4), ((3, 40, 5), 5),
    ((23, 9, 31), 12), ((17, 2), 1), ((40, 33), 6), ((70, 66, 70), 2)])
def test_fused_inference_matches_its_parts(cells, G):
    op, pred, prev, cur = setup(cells, G)
    want, top2, ls = parts(pred, prev, cur)
    got = torch.full_like(cur, float("nan"))
    pred.top2.zero_()
    pred.lscale.zero_()
    pred.predict(prev, cur, 1e-3, got)
    base = 2.0 * cur - prev
    corr = (want - base).abs().max().item()
    assert corr > 0.0 and torch.isfinite(got).all()
    assert (got - want).abs().max().item() <= 2.0 ** -5 * corr
    assert torch.equal(pred.top2, top2)
    # the same 135 FP64 squares in another order, then rounded to FP32
    assert ((pred.lscale - ls).abs() <= 1.2e-7 * ls).all()
    # components without an output are the plain extrapolation, bit for bit
    nc = G + 2
    plain = torch.ones(op.n_nodes, nc, dtype=torch.bool, device=cur.device)
    plain[:, :2] = False
    plain.scatter_(1, 2 + top2.long(), False)
    assert torch.equal(got.view(-1, nc)[plain], base.view(-1, nc)[plain])


def test_fused_inference_not_in_place():
    op, pred, prev, cur = setup((9, 8, 7), 3)
    want, _, _ = parts(pred, prev, cur)
    pred.predict(prev, cur, 1e-3, torch.empty_like(cur))
    x = cur.clone()
    pred.predict(prev, x, 1e-3, x)           # kernel by kernel
    assert torch.equal(x, want)
    arr = ctypes.c_void_p * 4
    p = ctypes.c_void_p
    with pytest.raises(HpsError):
        check(lib().hps_mlp_infer(
            op.handle, p(prev.data_ptr()), p(cur.data_ptr()), 1e-3, 1e3, 1.0,
            arr(*[w.data_ptr() for w in pred.mlp.Wb]), arr(*[b.data_ptr() for b in pred.mlp.b]),
            p(pred.out_scale.data_ptr()), p(pred.top2.data_ptr()), p(pred.lscale.data_ptr()),
            p(cur.data_ptr()), p(pred._ws.data_ptr())))


# 32 nodes per workgroup: fewer, a remainder, a mesh of one node plane
@pytest.mark.parametrize("cells,G", [((1, 1, 1), 1), ((7, 5, 9), 4), ((9, 10, 4), 12),
                                     ((31, 6), 3)])
def test_rows_of_a_prediction(cells, G):
    """X after predict holds that prediction's feature rows, bit for bit those
    of features(): asked for afterwards, with the inputs overwritten in
    between, and as a tensor that the program already holds"""
    op, pred, prev, cur = setup(cells, G)
    other = LearnedPredictor(op, pred.mlp, dt_scale=1e3)
    out = torch.empty_like(cur)
    want, _ = other.features(prev, cur, 1e-3)
    want = want.clone()
    pred.predict(prev, cur, 1e-3, out)
    prev2, cur2 = prev * 0.9, cur * 1.01
    prev.fill_(7.0)
    cur.fill_(5.0)
    rows = pred.X
    assert torch.isfinite(rows).all() and torch.equal(rows, want)
    want2, _ = other.features(prev2, cur2, 2e-3)
    pred.predict(prev2, cur2, 2e-3, out)
    assert pred.X is rows and torch.equal(rows, want2)
    mine = torch.zeros_like(rows)
    pred.X = mine
    pred.predict(prev2, cur2, 2e-3, out)
    assert torch.equal(mine, want2)


@pytest.mark.parametrize("n", [1, 255, 256, 524289])
def test_norm2_diff(n):
    op, _, _, _ = setup((3, 3, 3), 1)
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal(n), rng.standard_normal(n)
    r = ctypes.c_double()
    dx, dy = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    check(lib().hps_norm2_diff(op.handle, n, ctypes.c_void_p(dx.data_ptr()),
                               ctypes.c_void_p(dy.data_ptr()), ctypes.byref(r)))
    ref = np.linalg.norm(x - y)
    assert abs(r.value - ref) <= 1e-12 * ref
