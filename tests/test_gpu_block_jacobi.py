"""Node-block assembly and inversion for every component count.

The inverse is checked against the blocks the library returns: y = B^-1 x
computed through an explicit inverse has a residual |B y - x| of at most a
few nc eps cond(B) |B| |y| (elimination with partial pivoting, growth of
order one for these sizes; 16 allows for it).  Small time weights make the
mu row of the c column the larger one, so every block exchanges rows; large
ones leave the pivots on the diagonal.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from hpsint_amd import CartesianMesh, MobilityParams, SinteringOperatorGeneric  # noqa: E402
from hpsint_amd.operator import Preconditioner  # noqa: E402

EPS = np.finfo(np.float64).eps


def operator(cells, G, tensorial=False, degree=1, w0=1e3, h=0.5):
    mesh = CartesianMesh(cells, (0.0,) * len(cells), tuple(h * c for c in cells))
    op = SinteringOperatorGeneric(mesh, G, mobility=MobilityParams(tensorial=tensorial),
                                  fe_degree=degree)
    op.set_time_weights(w0, (-w0,))
    u = np.random.default_rng(G).uniform(0, 1, op.n_dofs)
    op.fill_quadrature_point_values(torch.from_numpy(u).cuda())
    return op


@pytest.mark.parametrize("w0", [1e3, 1e-3])
@pytest.mark.parametrize("G", range(1, 13))
def test_inverse_of_node_blocks(G, w0):
    op = operator((5, 4, 3), G, w0=w0)
    nc = G + 2
    B = op.node_blocks().cpu().numpy()
    x = np.random.default_rng(7).uniform(-1, 1, op.n_dofs)
    p = Preconditioner(op, "InverseComponentBlockDiagonalMatrix")
    p.do_update()
    y = op.initialize_dof_vector()
    p.vmult(y, torch.from_numpy(x).cuda())
    y = y.cpu().numpy().reshape(-1, nc)
    res = np.linalg.norm(np.einsum("nij,nj->ni", B, y) - x.reshape(-1, nc), axis=1)
    bound = 16 * nc * EPS * np.linalg.cond(B) * np.linalg.norm(B, axis=(1, 2))
    assert np.all(res <= bound * np.linalg.norm(y, axis=1))
    if w0 < 1.0:   # the case is what it claims: rows are exchanged
        assert np.all(np.abs(B[:, 1, 0]) > np.abs(B[:, 0, 0]))


# windows of 7 x 7 completed nodes, marches of 4 planes or more, cache tiles
# of 8 x 4 x 16 cells
@pytest.mark.parametrize("cells,G", [
    ((1, 1, 1), 1), ((6, 6, 3), 2), ((7, 13, 5), 3), ((9, 3, 17), 4), ((14, 5, 4), 5),
    ((8, 4, 16), 6), ((5, 8, 33), 7), ((20, 15, 18), 8), ((13, 7, 2), 9), ((3, 9, 7), 10),
    ((6, 2, 9), 11), ((8, 12, 6), 12)])
def test_one_pass_blocks_match_column_by_column(cells, G):
    """the cut-off operator with every order parameter active assembles the
    same blocks by applying the tangent to one unit input per column; both
    add the same products in other orders, at most 8 cells of 8 points"""
    op = operator(cells, G)
    nc = G + 2
    blocks = torch.empty(op.n_nodes, nc, nc, dtype=torch.float64, device="cuda")
    from hpsint_amd._ffi import check, lib
    import ctypes

    def get(fp32):
        Preconditioner(op, "InverseComponentBlockDiagonalMatrix").do_update(fp32=fp32)
        check(lib().hps_precond_get_blocks(op.handle, ctypes.c_void_p(blocks.data_ptr())))
        return blocks.clone()

    one64, one32 = get(False), get(True)
    u = torch.from_numpy(np.random.default_rng(G).uniform(0, 1, op.n_dofs)).cuda()
    op.set_grain_cut_off(1e-300)
    op.set_component_mask(u)
    op.fill_quadrature_point_values(u)
    col64 = get(False)
    scale = col64.abs().amax(dim=(1, 2), keepdim=True)
    assert ((one64 - col64).abs() <= 64 * EPS * scale * nc).all()
    eps32 = float(np.finfo(np.float32).eps)
    assert ((one32 - col64).abs() <= 64 * eps32 * scale * nc).all()
