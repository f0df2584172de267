"""Learned Newton initial-guess predictor (build-only; fills the predictor
slot of the driver, S/driver.h:2002-2050 with S/ =
applications/sintering/include/pf-applications/sintering/).

Network: per node, 272 inputs (27-node stencil of c, mu, sum eta^2 and the
node's top-2 order parameters, at t_n and as the scaled increment
t_n - t_{n-1}, plus dt) -> tanh hidden layers of width 128 -> 4 outputs, the
correction of the linear extrapolation 2 u_n - u_{n-1} on (c, mu, eta_top1,
eta_top2).  All arithmetic runs in the library's BF16-MFMA kernels (FP32
accumulation); torch tensors only hold the memory.  The plain Newton solve
from the predicted guess keeps the same tolerance, so the plain method stays
both the fallback and the reference for the result.
"""
import ctypes
import math

import torch

from ._ffi import HpsMlpParams, check, lib

N_IN = 272
N_OUT = 4


# the methods that the fused calls stand for
_OWN = {}


def _unchanged(obj, cls):
    """obj is a cls whose methods behind the fused calls are the class's own: a
    subclass or a program that replaces one of them gets it called"""
    return isinstance(obj, cls) and all(
        getattr(getattr(obj, name), "__func__", None) is f for name, f in _OWN[cls].items())


def _p(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


class MLP:
    """weights W_l (out x in, FP32 master + bf16 copy), biases b_l (FP32)"""

    def __init__(self, op, dims=(N_IN, 128, 128, 128, N_OUT), seed=0, device="cuda"):
        self.op = op
        self.dims = list(dims)
        g = torch.Generator(device="cpu").manual_seed(seed)
        self.W, self.Wb, self.b, self.mW, self.vW, self.mb, self.vb = [], [], [], [], [], [], []
        for l in range(len(dims) - 1):
            n_in, n_out = dims[l], dims[l + 1]
            bound = 1.0 / math.sqrt(n_in)
            w = (torch.rand(n_out, n_in, generator=g, dtype=torch.float64) * 2 - 1) * bound
            if l == len(dims) - 2:
                w *= 0.01   # start close to the plain linear extrapolation
            w = w.float().to(device)
            self.W.append(w)
            self.Wb.append(w.to(torch.bfloat16))
            self.b.append(torch.zeros(n_out, dtype=torch.float32, device=device))
            for lst in (self.mW, self.vW):
                lst.append(torch.zeros_like(w))
            for lst in (self.mb, self.vb):
                lst.append(torch.zeros(n_out, dtype=torch.float32, device=device))
        self.step = 0
        self._ws = {}

    @property
    def n_layers(self):
        return len(self.dims) - 1

    def _buf(self, key, shape, dtype):
        t = self._ws.get(key)
        if t is None or t.numel() < math.prod(shape) or t.dtype != dtype:
            t = torch.empty(math.prod(shape), dtype=dtype, device=self.W[0].device)
            self._ws[key] = t
        return t[:math.prod(shape)].view(*shape)

    def _gemm(self, ta, tb, epi, M, N, K, A, lda, B, ldb, C, ldc, bias=None, H=None, split=1):
        check(lib().hps_mlp_gemm(self.op.handle, ta, tb, epi, M, N, K, _p(A), lda, _p(B), ldb,
                                 _p(C), ldc, _p(bias), _p(H), split))

    def forward(self, X, M):
        """X: (M, 272) bf16 -> Y (M, 4) FP32; keeps the activations"""
        acts = [X]
        h = X
        for l in range(self.n_layers):
            n_in, n_out = self.dims[l], self.dims[l + 1]
            last = l == self.n_layers - 1
            out = self._buf(("h", l), (M, n_out), torch.float32 if last else torch.bfloat16)
            self._gemm(0, 1, 2 if last else 1, M, n_out, n_in, h, n_in, self.Wb[l], n_in, out,
                       n_out, bias=self.b[l])
            acts.append(out)
            h = out
        return acts[-1], acts

    def backward(self, acts, dY, M, split=None):
        """dY: (M, 4) bf16 -> gradients (gW, gb) per layer"""
        split = split or max(1, min(64, M // 2048))
        gW, gb = [None] * self.n_layers, [None] * self.n_layers
        dZ = dY
        for l in range(self.n_layers - 1, -1, -1):
            n_in, n_out = self.dims[l], self.dims[l + 1]
            A = acts[l]
            part = self._buf(("part", l), (split, n_out, n_in), torch.float32)
            self._gemm(1, 0, 0, n_out, n_in, M, dZ, n_out, A, n_in, part, n_in, split=split)
            g = self._buf(("gW", l), (n_out, n_in), torch.float32)
            check(lib().hps_mlp_sum_splits(self.op.handle, n_out * n_in, split, _p(part), _p(g)))
            gbl = self._buf(("gb", l), (n_out,), torch.float32)
            check(lib().hps_mlp_colsum(self.op.handle, M, n_out, _p(dZ), _p(gbl)))
            gW[l], gb[l] = g, gbl
            if l > 0:
                dA = self._buf(("dz", l), (M, n_in), torch.bfloat16)
                self._gemm(0, 0, 3, M, n_in, n_out, dZ, n_out, self.Wb[l], n_in, dA, n_in,
                           H=acts[l])
                dZ = dA
        return gW, gb

    def loss_grad(self, Y, T, M):
        dY = self._buf("dY", (M, N_OUT), torch.bfloat16)
        nb = 256
        part = self._buf("lpart", (nb,), torch.float32)
        loss = ctypes.c_float()
        check(lib().hps_mlp_loss(self.op.handle, M * N_OUT, _p(Y), _p(T), _p(dY), _p(part), nb,
                                 ctypes.byref(loss)))
        return loss.value, dY

    def adam(self, gW, gb, lr, b1=0.9, b2=0.999, eps=1e-8):
        self.step += 1
        for l in range(self.n_layers):
            n_in, n_out = self.dims[l], self.dims[l + 1]
            check(lib().hps_mlp_adam(self.op.handle, n_out, n_in, _p(self.W[l]), _p(self.mW[l]),
                                     _p(self.vW[l]), _p(gW[l]), lr, b1, b2, eps, self.step,
                                     _p(self.Wb[l])))
            check(lib().hps_mlp_adam(self.op.handle, 1, n_out, _p(self.b[l]), _p(self.mb[l]),
                                     _p(self.vb[l]), _p(gb[l]), lr, b1, b2, eps, self.step,
                                     None))

    def _train_fused(self, X, T, M, lr, b1=0.9, b2=0.999, eps=1e-8):
        """hps_mlp_train_step, or None where it does not cover the call:
        other widths, more rows than it takes, unaligned operands or a method
        of its own for a part of the step"""
        if not _unchanged(self, MLP) or self.dims != [N_IN, 128, 128, 128, N_OUT]:
            return None
        n = ctypes.c_int64()
        check(lib().hps_mlp_train_workspace(self.op.handle, M, ctypes.byref(n)))
        if n.value == 0 or any(t.data_ptr() % 16 for t in [X] + self.Wb):
            return None
        ws = self._buf("train", (n.value,), torch.uint8)
        p = HpsMlpParams(*[(ctypes.c_void_p * 4)(*[t.data_ptr() for t in ts])
                           for ts in (self.W, self.Wb, self.b, self.mW, self.vW, self.mb, self.vb)])
        loss = ctypes.c_float()
        check(lib().hps_mlp_train_step(self.op.handle, M, _p(X), _p(T), ctypes.byref(p), lr, b1,
                                       b2, eps, self.step + 1, _p(ws), ctypes.byref(loss)))
        self.step += 1
        return loss.value

    def train_step(self, X, T, M, lr):
        loss = self._train_fused(X, T, M, lr)
        if loss is not None:
            return loss
        Y, acts = self.forward(X, M)
        loss, dY = self.loss_grad(Y, T, M)
        gW, gb = self.backward(acts, dY, M)
        self.adam(gW, gb, lr)
        return loss


class LearnedPredictor:
    """Newton initial guess u_pred = 2 u_n - u_{n-1} + ls * out_scale * MLP(features).

    ls is each node's local increment scale (RMS of the stencil increments
    of u_n - u_{n-1}, computed by the feature kernel); increment features are
    divided by it and the outputs multiplied by it, so the network sees the
    same scales in the quiet bulk and at moving interfaces.  out_scale holds
    one global constant per output, fixed at training."""

    def __init__(self, op, mlp: MLP = None, dt_scale=1.0, out_scale=None):
        self.op = op
        self.mlp = mlp or MLP(op)
        self.dt_scale = dt_scale
        dev = self.mlp.W[0].device
        self.out_scale = torch.tensor(list(out_scale) if out_scale is not None else [1.0] * N_OUT,
                                      dtype=torch.float32, device=dev)
        n = op.n_nodes
        self._X = None
        self._ws = None
        self._inferred = None   # dt and scales of the last fused prediction
        self.top2 = torch.empty(n, 2, dtype=torch.int32, device=dev)
        self.lscale = torch.empty(n, dtype=torch.float32, device=dev)
        self.use_network = True
        self.inc_scale = 1.0

    @property
    def X(self):
        """feature rows of the last features() or predict() call.  The fused
        inference forms them in registers: they are written when they are first
        asked for, and from then on by each prediction"""
        if self._X is None:
            self._X = torch.empty(self.op.n_nodes, N_IN, dtype=torch.bfloat16,
                                  device=self.mlp.W[0].device)
            if self._inferred is not None:
                self._write_rows()
        return self._X

    @X.setter
    def X(self, rows):
        self._X = rows

    def _write_rows(self):
        check(lib().hps_mlp_infer_rows(self.op.handle, *self._inferred, _p(self.top2),
                                       _p(self._ws), _p(self._X)))

    def step_scale(self, u_prev, u_cur):
        """RMS of u_cur - u_prev, computed by the library"""
        n = self.op.n_dofs
        r = ctypes.c_double()
        check(lib().hps_norm2_diff(self.op.handle, n, _p(u_cur), _p(u_prev), ctypes.byref(r)))
        return max(r.value / math.sqrt(n), 1e-300)

    def features(self, u_prev, u_cur, dt):
        self.inc_scale = 1.0 / self.step_scale(u_prev, u_cur)
        self._inferred = None
        check(lib().hps_mlp_features(self.op.handle, _p(u_prev), _p(u_cur), dt, self.dt_scale,
                                     self.inc_scale, _p(self.X), _p(self.top2),
                                     _p(self.lscale)))
        return self.X, self.top2

    def _infer_workspace(self, u_prev, u_cur, out):
        """the workspace of hps_mlp_infer, or None where that call does not
        cover the prediction: other widths than the built network's, a
        network or features() of the program's own, an output that overlaps an
        input (its stencils read the inputs while others' results are written)
        or a mesh beyond its 32-bit offsets"""
        size = 8 * self.op.n_dofs
        if (not _unchanged(self, LearnedPredictor) or not _unchanged(self.mlp, MLP)
                or self.mlp.dims != [N_IN, 128, 128, 128, N_OUT]
                or any(abs(out.data_ptr() - u.data_ptr()) < size for u in (u_prev, u_cur))):
            return None
        if self._ws is None:
            n = ctypes.c_int64()
            check(lib().hps_mlp_infer_workspace(self.op.handle, ctypes.byref(n)))
            self._ws = torch.empty(n.value, dtype=torch.uint8, device=self.mlp.W[0].device)
        return self._ws if self._ws.numel() else None

    def predict(self, u_prev, u_cur, dt, out):
        Y = None
        ws = self._infer_workspace(u_prev, u_cur, out) if self.use_network else None
        if ws is not None:
            self.inc_scale = 1.0 / self.step_scale(u_prev, u_cur)
            arr = ctypes.c_void_p * self.mlp.n_layers
            check(lib().hps_mlp_infer(
                self.op.handle, _p(u_prev), _p(u_cur), dt, self.dt_scale, self.inc_scale,
                arr(*[w.data_ptr() for w in self.mlp.Wb]),
                arr(*[b.data_ptr() for b in self.mlp.b]), _p(self.out_scale), _p(self.top2),
                _p(self.lscale), _p(out), _p(ws)))
            self._inferred = (dt, self.dt_scale, self.inc_scale)
            if self._X is not None:
                self._write_rows()
            return out
        if self.use_network:
            X, _ = self.features(u_prev, u_cur, dt)
            Y, _ = self.mlp.forward(X, self.op.n_nodes)
        check(lib().hps_mlp_predict(self.op.handle, _p(u_prev), _p(u_cur), _p(Y),
                                    _p(self.top2), _p(self.out_scale), _p(self.lscale),
                                    _p(out)))
        return out

    def targets(self, u_prev, u_cur, u_next, T):
        """(u_next - (2 u_cur - u_prev)) / (ls * out_scale) on the 4 outputs;
        call after features() of the same (u_prev, u_cur)"""
        check(lib().hps_mlp_targets(self.op.handle, _p(u_prev), _p(u_cur), _p(u_next),
                                    _p(self.top2), _p(self.out_scale), _p(self.lscale), _p(T)))
        return T

    def __call__(self, x, states, dt):
        """TimeStepper hook: states = [u_n, u_{n-1}, ...]"""
        if len(states) < 2:
            return x
        return self.predict(states[1], states[0], dt, x)


_OWN.update({
    MLP: {n: getattr(MLP, n) for n in ("forward", "loss_grad", "backward", "adam")},
    LearnedPredictor: {"features": LearnedPredictor.features},
})
