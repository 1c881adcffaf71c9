"""Launch shapes chosen for one kernel of an operator that has been used: general (SELL) storage follows the row blocks of
the application, whose default depends on the caller's choice for the vector kernels too.  Products are compared with
those before (row sums do not depend on the blocks: the same bits) and with the CSR matrix in scipy, whose sums of at
most 27 terms in the same order differ by fused roundings only; solutions through their residual against the CSR matrix
(the solver stops at 1e-10 of its own residual; 2e-10 leaves room for the round-off between the two)."""
import numpy as np
import pytest
import torch

from problems import hgdt_problem

pytestmark = pytest.mark.gpu


def _operator(H, case):
    if case == "batch":
        grid = H.Grid.union([H.Grid.structured("quad", [0, 0], [1, 1], [m, m]) for m in (5, 70, 33, 131)])
    elif case == "mesh":
        g = H.Grid.structured("tri", [0, 0], [1, 1], [211, 160])
        perm = np.random.default_rng(3).permutation(len(g.coordinates())).astype(np.int32)
        coords = np.empty_like(g.coordinates())
        coords[perm] = g.coordinates()
        grid = H.Grid.from_arrays("tri", coords, perm[g.connectivity()])
    else:
        grid = H.Grid.structured("quad", [0, 0], [1, 1], [400, 351])
    kappa = torch.from_numpy(H.fields.lognormal(7, grid.num_elements)).cuda()
    space, op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=grid)[1:]
    op.set_format("sell64")
    op.assemble()
    return space, op


@pytest.mark.parametrize("first", ["apply", "apply_inverse"])
@pytest.mark.parametrize("case", ["quads", "batch", "mesh"])
def test_vector_shape_of_a_used_operator(hgdt_mod, case, first):
    H = hgdt_mod
    print(f"case {case}, used by {first}", flush=True)
    space, op = _operator(H, case)
    A, b = op.matrix.to_scipy(), op.rhs.cpu().numpy()
    v = torch.from_numpy(H.fields.uniform(8, space.num_DoFs)).cuda()
    y = A @ v.cpu().numpy()
    scale = abs(A) @ np.abs(v.cpu().numpy())
    before = op.apply(v) if first == "apply" else None
    if before is None:
        op.apply_inverse("rhs")
        assert op.solve_workgroups() > 0
        before = op.apply(v)
    blocks = [op.get_launch(3), op.get_launch(4)]
    if first == "apply_inverse":  # the shapes of the solve in one launch (made for the first solve)
        assert blocks[0] == blocks[1] and blocks[0][0] == 512
    for shape in (blocks[1], (256, 4), (512, 1), (64, 1), blocks[1]):
        print(f"  vector kernels {shape}", flush=True)
        op.set_launch(4, *shape)
        got = op.apply(v)
        assert torch.equal(got, before)
        assert np.all(np.abs(got.cpu().numpy() - y) <= 30 * np.finfo(float).eps * scale)
        x = op.apply_inverse("rhs").cpu().numpy()
        assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)
        assert torch.equal(op.apply(v), before)
    # the application's blocks again, then the next assembly
    op.set_launch(3, 128, 2)
    assert torch.equal(op.apply(v), before)
    op.assemble()
    x = op.apply_inverse("rhs").cpu().numpy()
    assert np.linalg.norm(b - A @ x) <= 2e-10 * np.linalg.norm(b)
    assert torch.equal(op.apply(v), before)


@pytest.mark.parametrize("shapes", [None, ((256, 1), (256, 1))])
def test_column_staging_asked_for(hgdt_mod, shapes):
    """mode 1 runs the staged application (kernels per iteration) wherever it applies, also where the solve would be one
    launch; the other modes leave that to the size; storage without diagonals has nothing to stage"""
    H = hgdt_mod
    print(f"case column staging {shapes}", flush=True)
    kappa = torch.from_numpy(H.fields.lognormal(7, 150 * 131)).cuda()
    op = hgdt_problem(H, "heat_q1", [150, 131], kappa)[2]
    if shapes:
        op.set_launch(3, *shapes[0])
        op.set_launch(4, *shapes[1])
    op.assemble()
    xs = []
    for mode in (1, 0, 1, -1):
        op.set_column_staging(mode)
        xs.append(op.apply_inverse("rhs"))
        assert op.last_solve["column_staged"] == (mode == 1), mode
        assert (op.solve_workgroups() == 0) == (mode == 1), mode
    assert torch.equal(xs[0], xs[2]) and torch.equal(xs[1], xs[3])
    if shapes:
        assert torch.equal(xs[0], xs[1])
    op.set_column_staging(1)
    op.set_format("sell64")
    op.apply_inverse("rhs")
    assert op.last_solve["column_staged"] == 0
    assert shapes or op.solve_workgroups() > 0  # (general storage in one launch: blocks of 512 lanes)
