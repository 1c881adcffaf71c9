"""Symmetric discontinuous forms evaluated straight into the rows of the matrix against the staged blocks, which an operator
on a caller's matrix always uses.  An entry is a sum of at most 5 contributions of at most 6 terms, from geometries
of some ten operations each: both ways stay within 100 roundings (1e-14) of the exact sum, relative to the largest
entry of the row; bound 1e-13."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _grid(H, geometry, cells, scattered):
    grid = H.Grid.structured(geometry, [0.] * len(cells), [1., 0.8, 1.3][:len(cells)], cells)
    if not scattered:
        return grid
    X, conn = grid.coordinates(), grid.connectivity()
    rng = np.random.default_rng(4)
    X = X + 0.1 / max(cells) * rng.uniform(-1, 1, X.shape)
    vp, ep = rng.permutation(len(X)), rng.permutation(len(conn))
    Y = np.empty_like(X)
    Y[vp] = X
    return H.Grid.from_arrays(geometry, Y, vp[conn][ep].astype(np.int32))


def _operator(H, grid, forms, matrix=None):
    kappa = torch.from_numpy(H.fields.lognormal(2, grid.num_elements)).cuda()
    omega = torch.from_numpy(H.fields.lognormal(3, grid.num_elements)).cuda()
    space = H.DiscontinuousLagrangeSpace(grid, 1)
    op = H.make_matrix_operator(space, H.Stencil.element_and_intersection, matrix=matrix)
    if "e" in forms:
        op.append(H.LocalElementIntegralBilinearForm(H.LocalLaplaceIntegrand(kappa)))
        op.append(H.LocalElementIntegralBilinearForm(H.LocalProductIntegrand(2.0)))
    op.append(H.LocalCouplingIntersectionIntegralBilinearForm(
        H.LocalLaplaceIPDGInnerCoupling(1.0, kappa, omega) + H.LocalIPDGInnerPenalty(16.0, omega)), {},
        H.ApplyOn.InnerIntersectionsOnce())
    if "b" in forms:
        op.append(H.LocalIntersectionIntegralBilinearForm(
            H.LocalIPDGBoundaryPenalty(16.0, omega) + H.LocalLaplaceIPDGDirichletCoupling(1.0, kappa)), {},
            H.ApplyOn.CustomBoundaryIntersections(H.AllDirichletBoundaryInfo()))
    op.assemble()
    return op


@pytest.mark.parametrize("geometry,cells,scattered", [
    ("quad", [1, 1], False), ("quad", [2, 1], False), ("quad", [9, 8], False), ("quad", [64, 33], False),
    ("tri", [1, 1], False), ("tri", [7, 9], False), ("tri", [11, 6], True), ("tet", [1, 1, 1], False),
    ("tet", [3, 4, 5], False), ("tet", [5, 4, 3], True)])
@pytest.mark.parametrize("forms", ["eb", "e", "b", ""])
def test_rows_equal_staged_blocks(hgdt_mod, geometry, cells, scattered, forms):
    print(f"case rows {geometry} {cells} {scattered} {forms}", flush=True)
    H = hgdt_mod
    grid = _grid(H, geometry, cells, scattered)
    A = _operator(H, grid, forms).matrix
    zero = H.CsrMatrix(A.row_ptr, A.cols, torch.zeros_like(A.values), A.shape)
    B = _operator(H, grid, forms, matrix=zero).matrix.to_scipy()
    A = A.to_scipy()
    assert A.nnz == B.nnz
    scale = np.maximum(abs(B).max(axis=1).toarray().ravel(), 1e-300)
    err = abs(A - B).max(axis=1).toarray().ravel() / scale
    print(f"  {grid.num_elements} elements, largest difference {err.max():.1e} of its row")
    assert err.max() <= 1e-13
    assert abs(A - A.T).max() == 0.0
