"""The fused training step (hps_mlp_train_step) against the layer-by-layer
kernels: the same roundings to bf16 (activations, dY, gradients between
layers), other FP32 accumulation orders, so an activation or a gradient may
round to the neighbouring bf16 value; the bound of 5e-3 in relative l2 is the
one that the layer-by-layer kernels keep against the numpy restatement."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from hpsint_amd import CartesianMesh, SinteringOperatorGeneric  # noqa: E402
from hpsint_amd.predictor import MLP, N_IN, N_OUT  # noqa: E402


def network(op):
    mlp = MLP(op, seed=2)
    g = torch.Generator(device="cuda").manual_seed(9)
    mlp.W[-1].normal_(0, 0.1, generator=g)
    mlp.Wb[-1].copy_(mlp.W[-1])
    for t in mlp.b + mlp.mW + mlp.mb:
        t.uniform_(-0.1, 0.1, generator=g)
    for t in mlp.vW + mlp.vb:
        t.uniform_(0.5, 1.0, generator=g)
    mlp.step = 50
    return mlp


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


# 64 rows per workgroup, splits of 512 rows (more from 16384 rows on)
@pytest.mark.parametrize("M", [1, 63, 64, 65, 511, 1025, 3000, 20000])
def test_fused_step_matches_layer_by_layer(M):
    op = SinteringOperatorGeneric(CartesianMesh((4, 4, 4), (0, 0, 0), (4.0, 4.0, 4.0)), 2)
    rng = np.random.default_rng(M)
    X = torch.from_numpy(rng.uniform(-1, 1, (M, N_IN)).astype(np.float32)).cuda().bfloat16()
    T = torch.from_numpy(rng.uniform(-1, 1, (M, N_OUT)).astype(np.float32)).cuda()
    one, ref = network(op), network(op)
    before = [t.clone() for t in ref.W + ref.b + ref.mW + ref.mb]
    Y, acts = ref.forward(X, M)
    want, dY = ref.loss_grad(Y, T, M)
    gW, gb = ref.backward(acts, dY, M)
    ref.adam(gW, gb, 1e-3)
    got = one._train_fused(X, T, M, 1e-3)
    assert got is not None and one.step == ref.step
    assert abs(got - want) <= 5e-3 * want
    after1 = one.W + one.b + one.mW + one.mb
    after2 = ref.W + ref.b + ref.mW + ref.mb
    for k, (t0, a, b) in enumerate(zip(before, after1, after2)):
        decay = 0.9 if k >= 8 else 1.0          # moments: 0.9 m + 0.1 g
        assert rel(a - decay * t0, b - decay * t0) < 5e-3, k
    for a, w in zip(one.Wb, one.W):
        assert torch.equal(a, w.bfloat16())


def test_other_widths_keep_the_layer_kernels():
    op = SinteringOperatorGeneric(CartesianMesh((4, 4, 4), (0, 0, 0), (4.0, 4.0, 4.0)), 2)
    mlp = MLP(op, dims=(N_IN, 64, N_OUT), seed=0)
    X = torch.rand(100, N_IN, device="cuda").bfloat16()
    T = torch.rand(100, N_OUT, device="cuda")
    assert mlp._train_fused(X, T, 100, 1e-3) is None
    first = mlp.train_step(X, T, 100, 1e-3)
    assert np.isfinite(first) and mlp.step == 1
