"""Reductions whose grid follows the vector's length, and the tile depth that
follows the mesh, at the edges of their rules."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from hpsint_amd import _ffi  # noqa: E402
from hpsint_amd.operator import (CartesianMesh, FreeEnergyParams, MobilityParams,  # noqa: E402
                                 SinteringOperatorGeneric)

pytestmark = pytest.mark.gpu


def dev(x, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=dtype).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy().astype(np.float64)


# one block, one block and its neighbour, the last length of a growing grid,
# the full grid with and without a remainder
@pytest.mark.parametrize("n", [1, 511, 512, 513, 1025, 2048 * 512, 2048 * 512 + 1, 3000001])
@pytest.mark.parametrize("k", [1, 16, 17, 31])
def test_reductions_at_the_edges_of_the_grid_rule(n, k):
    """A sum of FP64 products: a thread adds at most n / 2^19 + 2 of them, then
    17 levels of trees and rows follow, each rounding at most half an ulp
    (2^-53) of the sum of magnitudes: 32 + n / 2^19 halves.  An update w -=
    sum h_j V_j rounds once per product and once per sum: 2 k + 2 halves of the
    storage type, relative to the magnitudes."""
    mesh = CartesianMesh((2, 2, 2), (0, 0, 0), (2.0, 2.0, 2.0))
    op = SinteringOperatorGeneric(mesh, 1)
    h, L = op.handle, _ffi.lib()
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    rng = np.random.default_rng(n + k)
    tol = (32 + n / 2**19) * 2.0**-53
    r = ctypes.c_double()
    hh = (ctypes.c_double * k)()
    for dtype, npt, ulp, suf in ((torch.float64, np.float64, 2.0**-53, ""),
                                 (torch.float32, np.float32, 2.0**-24, "_f32")):
        V = rng.standard_normal((k, n)).astype(npt)
        w = rng.standard_normal(n).astype(npt)
        V64, w64 = V.astype(np.longdouble), w.astype(np.longdouble)
        dV, dw = dev(V.ravel(), dtype), dev(w, dtype)
        _ffi.check(getattr(L, "hps_norm2" + suf)(h, n, P(dw), ctypes.byref(r)))
        ref = np.sqrt(np.sum(w64 * w64))
        assert abs(r.value - ref) <= tol * ref
        _ffi.check(getattr(L, "hps_multi_dot" + suf)(h, n, k, P(dV), P(dw), hh))
        for j in range(k):
            ref, mag = np.sum(V64[j] * w64), np.sum(np.abs(V64[j] * w64))
            assert abs(hh[j] - ref) <= tol * mag, (j, hh[j], ref)
        _ffi.check(getattr(L, "hps_multi_axpy_norm" + suf)(h, n, k, P(dV), hh, P(dw),
                                                          ctypes.byref(r)))
        c = np.array(list(hh), dtype=np.longdouble)
        ref, mag = w64 - c @ V64, np.abs(w64) + np.abs(c) @ np.abs(V64)
        got = host(dw)
        assert np.all(np.abs(got - ref) <= (2 * k + 2) * ulp * mag)
        nrm = np.sqrt(np.sum(got.astype(np.longdouble)**2))
        # (n = 1: everything cancels and the norm is of rounding errors)
        slack = tol * nrm + (2 * k + 2) * ulp * np.sqrt(np.sum(mag**2))
        assert abs(r.value - nrm) <= slack


def orthonormal(rng, k, n, npt):
    """k orthonormal rows (n >= k; for fewer entries any rows)"""
    V = rng.standard_normal((k, n))
    if n >= k:
        V = np.linalg.qr(V.T)[0].T
    return np.ascontiguousarray(V).astype(npt)


def call_orthogonalise(op, V, w, dtype):
    k, n = V.shape
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    dV, dw = dev(V.ravel(), dtype), dev(w, dtype)
    h, r = (ctypes.c_double * k)(), ctypes.c_double()
    f = "hps_orthogonalise" + ("_f32" if dtype == torch.float32 else "")
    _ffi.check(getattr(_ffi.lib(), f)(op.handle, n, k, P(dV), P(dw), h, ctypes.byref(r)))
    return np.array(list(h), dtype=np.longdouble), r.value, host(dw)


# up to 256 reduction blocks (131072 entries) the partial sums are summed in the
# consuming kernels, beyond that in kernels of their own; k in passes of 16
@pytest.mark.parametrize("n,k", [(1, 1), (1, 17), (511, 16), (512, 31), (513, 1), (513, 32),
                                 (131072, 1), (131072, 16), (131072, 31), (131073, 1),
                                 (131073, 17), (131073, 32), (2048 * 512 + 1, 16),
                                 (2048 * 512 + 1, 31)])
@pytest.mark.parametrize("near", [False, True])   # near: a second pass is due
def test_orthogonalise(n, k, near):
    """h, the norm and the normalised w of the Gram-Schmidt step that GMRES runs
    on.  A pass rounds w -= sum h_j V_j once per product and once per sum, 2 k +
    2 halves of the storage type's spacing of |w| + sum |h_j V_j|, and the
    normalisation twice more: with what it returned, sum_j h_j V_j + norm w is
    the old w to that, twice with two passes.  The dots' own errors (32 + n /
    2^19 halves in FP64) move h and w together and stay out of that sum; they
    and the roundings bound what is left along V."""
    op = SinteringOperatorGeneric(CartesianMesh((2, 2, 2), (0, 0, 0), (2.0,) * 3), 1)
    rng = np.random.default_rng(n + k)
    for dtype, npt, ulp in ((torch.float64, np.float64, 2.0**-53),
                            (torch.float32, np.float32, 2.0**-24)):
        tol = (32 + n / 2**19) * 2.0**-53
        V = orthonormal(rng, k, n, npt)
        w = rng.standard_normal(n)
        if near:
            w = 1e-2 * w / np.linalg.norm(w) + rng.uniform(0.5, 1, k) @ V.astype(np.float64)
        w = w.astype(npt)
        h, norm, got = call_orthogonalise(op, V, w, dtype)
        V64, w64 = V.astype(np.longdouble), w.astype(np.longdouble)
        passes = 2 if near else 1
        mag = np.abs(w64) + np.abs(h) @ np.abs(V64)
        left = np.abs(h @ V64 + norm * got.astype(np.longdouble) - w64)
        assert np.all(left <= passes * (2 * k + 2) * ulp * mag + 4 * ulp * norm * np.abs(got))
        if n < 2 * k:                     # (nothing or roundings left: only the sum)
            continue
        assert abs(np.sqrt(np.sum(got.astype(np.longdouble)**2)) - 1) <= tol + 2 * ulp
        along = np.abs(V64 @ got.astype(np.longdouble))
        lost = np.sqrt(np.sum(mag**2)) / norm if not near else 1.0
        assert np.all(along <= ((2 * k + 4) * ulp + tol) * max(1.0, float(lost))), along.max()


def test_orthogonalise_rounds_once_for_the_norm():
    """FP32 storage, two passes: w is rounded by each update and by one
    normalisation at the end.  The same steps in FP64 give the same FP32 numbers
    but where an FP64 rounding falls on a tie (far below one in a thousand); one
    rounding more changes about one number in six."""
    op = SinteringOperatorGeneric(CartesianMesh((2, 2, 2), (0, 0, 0), (2.0,) * 3), 1)
    for n, k in ((5000, 8), (200000, 5)):
        rng = np.random.default_rng(k)
        V = orthonormal(rng, k, n, np.float32)
        V64 = V.astype(np.float64)
        w = rng.standard_normal(n)
        w = (0.2 * w / np.linalg.norm(w) + rng.uniform(0.5, 1, k) @ V64).astype(np.float32)
        w1 = (w - (V64 @ w) @ V64).astype(np.float32).astype(np.float64)
        w2 = (w1 - (V64 @ w1) @ V64).astype(np.float32).astype(np.float64)
        want = (w2 / np.linalg.norm(w2)).astype(np.float32)
        _, norm, got = call_orthogonalise(op, V, w, torch.float32)
        assert abs(norm - np.linalg.norm(w2)) <= 1e-12 * norm
        same = np.mean(got.astype(np.float32) == want)
        # the entry a w is a times 1 / norm: a rounding in FP64 more
        assert same > 0.999, same


def test_orthogonalise_zero():
    """nothing left: norm 0 and w = 0, not NaN; k out of range is refused"""
    op = SinteringOperatorGeneric(CartesianMesh((2, 2, 2), (0, 0, 0), (2.0,) * 3), 1)
    for dtype, npt in ((torch.float64, np.float64), (torch.float32, np.float32)):
        for n in (7, 200000):
            V = np.zeros((2, n), npt)
            V[0, 0] = V[1, n - 1] = 1.0
            w = 3.0 * V[0] - 5.0 * V[1]
            h, norm, got = call_orthogonalise(op, V, w, dtype)
            assert list(h) == [3.0, -5.0] and norm == 0.0 and not got.any()
            h, norm, got = call_orthogonalise(op, V, 0 * w, dtype)
            assert list(h) == [0.0, 0.0] and norm == 0.0 and not got.any()
    with pytest.raises(_ffi.HpsError):
        call_orthogonalise(op, np.zeros((33, 8)), np.zeros(8), torch.float64)


# layers: the deepest of 16, 8, 4 and (up to 4 order parameters) 2 that gives 768
# tiles of 8 x 4 cells (2D: 64) and that many layers, or the shallowest
@pytest.mark.parametrize("cells,G,tens,layers", [
    ((24, 24, 24), 4, False, 2),    # fewest layers per tile
    ((24, 24, 24), 5, False, 4),    # fewest of five and more order parameters
    ((64, 40, 45), 3, False, 4),    # 960 tiles; 480 with 8 layers
    ((64, 64, 64), 4, False, 8),    # 1024; 512 with 16
    ((64, 64, 64), 7, False, 8),
    ((96, 96, 48), 2, False, 16),   # 864: unchanged
    ((160, 81), 2, False, 2), ((33, 500), 3, True, 2), ((17, 9, 30), 3, True, 2),
    ((2000, 368), 2, False, 8)])    # 32 columns, 46 rows of tiles; 23 with 16 layers
def test_tile_depth_of_small_meshes(monkeypatch, cells, G, tens, layers):
    """tangent, residual and diagonal with the depth chosen for the mesh: bit for
    bit those of the expected depth, and against 16 layers.  Only the order in
    which the cells of a node are added differs there: 8 (2D 4) cell sums, 8
    roundings of half an ulp of values that may cancel to about a tenth: 1e-14 in
    the norm"""
    dim = len(cells)
    mesh = CartesianMesh(cells, (0.0,) * dim, tuple(0.5 * c for c in cells))
    nn = int(np.prod([c + 1 for c in cells]))
    rng = np.random.default_rng(G)
    u = rng.uniform(0, 1, size=(nn, G + 2))
    src = rng.uniform(-1, 1, size=u.size)

    def results():
        op = SinteringOperatorGeneric(mesh, G, FreeEnergyParams(), MobilityParams(tensorial=tens))
        op.set_time_weights(1000.0, (-1000.0,))
        op.fill_quadrature_point_values(dev(u.ravel()))
        out = []
        for dtype in (torch.float64, torch.float32):
            dst = op.initialize_dof_vector(dtype)
            op.vmult(dst, dev(src, dtype))
            out.append(host(dst))
        dst = op.initialize_dof_vector()
        op.evaluate_nonlinear_residual(dst, dev(u.ravel()), 2, old=[dev(0.9 * u.ravel())])
        out.append(host(dst))
        inv = op.initialize_dof_vector()
        op.compute_inverse_diagonal(inv)
        out.append(host(inv))
        return out

    got = results()
    monkeypatch.setenv("HPSINT_AMD_TILE_M", str(layers))
    for g, r in zip(got, results()):
        assert np.array_equal(g, r)
    monkeypatch.setenv("HPSINT_AMD_TILE_M", "16")
    ref = results()
    assert layers == 16 or not np.array_equal(got[0], ref[0])
    for g, r, tol in zip(got, ref, (1e-14, 1e-14 * 2.0**29, 1e-14, 1e-14)):
        assert np.linalg.norm(g - r) <= tol * np.linalg.norm(r)
