"""Solves in one launch (vectors on the chip) against solves of three kernels per iteration, which a timed solve
(time_spmv) always issues: the same operations in the same order, so the bits, iteration counts and residuals
are equal.  Sizes: one row per lane and more, one workgroup and many, rows past the last full block, stencils that
reach over several workgroups, and operators too large or of a storage the launch does not take."""
import numpy as np
import pytest
import torch

from problems import hgdt_problem

pytestmark = pytest.mark.gpu


def _both(hgdt, op, **kw):
    x1 = op.apply_inverse("rhs", **kw)
    wg, s1, i1 = op.solve_workgroups(), dict(op.last_solve), op.instance_stats()
    x2 = op.apply_inverse("rhs", time_spmv=8, **kw)
    s2, i2 = dict(op.last_solve), op.instance_stats()
    assert op.solve_workgroups() == 0
    assert torch.equal(x1, x2)
    assert np.array_equal(i1[0], i2[0]) and np.array_equal(i1[1], i2[1])
    for k in ("iterations", "relres", "true_relres", "converged"):
        assert s1[k] == s2[k], k
    return wg


@pytest.mark.parametrize("kind,cells,workgroups", [
    ("heat_q1", [1, 1], 1), ("heat_q1", [2, 3], 1), ("heat_q1", [15, 15], 1), ("heat_q1", [22, 22], 1),
    ("heat_q1", [31, 15], 1), ("heat_q1", [63, 63], None), ("heat_q1", [90, 91], None), ("heat_q1", [700, 37], None),
    ("heat_q1", [3, 2000], None), ("heat_q1", [361, 362], None), ("heat_q1", [515, 509], None),
    ("p1_tets", [3, 2, 4], 1), ("p1_tets", [20, 17, 13], None), ("p1_tets", [9, 40, 31], None),
    ("p1_tets", [47, 48, 49], None), ("p1_tets", [86, 87, 88], 222), ("p1_tets", [120, 125, 60], 152),
    ("p1_tets", [127, 128, 127], None)])
def test_one_launch_equals_three_kernels(hgdt_mod, kind, cells, workgroups):
    print(f"case {kind} {cells}", flush=True)
    ne = int(np.prod(cells)) * (6 if kind == "p1_tets" else 1)
    kappa = torch.from_numpy(hgdt_mod.fields.lognormal(5, ne)).cuda()
    grid, space, op = hgdt_problem(hgdt_mod, kind, cells, kappa)
    op.assemble()
    wg = _both(hgdt_mod, op)
    print(f"  {space.num_DoFs} DoFs, {wg} workgroups, {op.last_solve['iterations']} iterations")
    assert wg > 0 and (workgroups is None or wg == workgroups)


@pytest.mark.parametrize("apply,vector,taken", [
    ((64, 1), (64, 1), True), ((1024, 1), (512, 1), True), ((128, 1), (256, 1), True), ((512, 2), (512, 2), True),
    ((512, 8), (512, 8), True), ((256, 1), (256, 4), False), ((512, 4), (512, 2), False), ((512, 1), (64, 8), False),
    ((256, 2), (256, 1), False), ((192, 1), (256, 1), False), ((256, 1), (1024, 1), False)])
def test_launch_shapes(hgdt_mod, apply, vector, taken):
    """shapes of the two row partitions: taken by the one launch (with the shape's bits) or not"""
    print(f"case shapes {apply} {vector}", flush=True)
    kappa = torch.from_numpy(hgdt_mod.fields.lognormal(6, 150 * 131)).cuda()
    grid, space, op = hgdt_problem(hgdt_mod, "heat_q1", [150, 131], kappa)
    op.set_launch(3, *apply)
    op.set_launch(4, *vector)
    op.assemble()
    assert (_both(hgdt_mod, op) > 0) == taken


def test_batch_initial_guess_and_limits(hgdt_mod):
    """uneven instances in one launch, a start from a given iterate, a stop at max_iter, a zero right-hand side"""
    H = hgdt_mod
    print("case batch", flush=True)
    sizes = [3, 150, 22, 64, 97]
    parts = [H.Grid.structured("quad", [0, 0], [1, 1], [m, m]) for m in sizes]
    union = H.Grid.union(parts)
    kappa = torch.from_numpy(H.fields.lognormal(7, union.num_elements)).cuda()
    grid, space, op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=union)
    op.assemble()
    assert _both(H, op) >= len(sizes)
    guess = torch.from_numpy(H.fields.uniform(8, space.num_DoFs)).cuda()
    got = []
    for spmv in (0, 8):
        got.append(op.apply_inverse("rhs", guess.clone(), opts={"initial_guess": True}, time_spmv=spmv))
    assert torch.equal(*got)
    for limit in (1, 2, 3, 40):
        xs = []
        for spmv in (0, 8):
            x = torch.zeros(space.num_DoFs, dtype=torch.float64, device="cuda")
            with pytest.raises(H.linear_solver_failed):
                op.apply_inverse("rhs", x, opts={"max_iter": limit}, time_spmv=spmv)
            assert op.last_solve["iterations"] == limit and not op.last_solve["converged"]
            xs.append(x)
        assert torch.equal(*xs)
    zero = torch.zeros(space.num_DoFs, dtype=torch.float64, device="cuda")
    x = op.apply_inverse(zero)
    assert op.solve_workgroups() > 0 and op.last_solve["iterations"] == 0 and torch.count_nonzero(x) == 0


def test_two_threads_two_streams(hgdt_mod):
    """solves of two operators from two threads on their own streams: each equal to its solve alone"""
    import threading

    print("case two threads", flush=True)
    ops, alone = [], []
    for seed, cells in ((11, [300, 280]), (12, [340, 200])):
        kappa = torch.from_numpy(hgdt_mod.fields.lognormal(seed, cells[0] * cells[1])).cuda()
        op = hgdt_problem(hgdt_mod, "heat_q1", cells, kappa)[2]
        op.assemble()
        alone.append(op.apply_inverse("rhs"))
        ops.append(op)
    torch.cuda.synchronize()
    got = [[], []]

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                got[k].append(ops[k].apply_inverse("rhs"))
        s.synchronize()

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    for k in range(2):
        assert len(got[k]) == 5 and all(torch.equal(x, alone[k]) for x in got[k])


def _poisson(H, geometry, order, cells, seed):
    grid = H.Grid.structured(geometry, [0.] * len(cells), [1.] * len(cells), cells)
    kappa = torch.from_numpy(H.fields.lognormal(seed, grid.num_elements)).cuda()
    space = H.ContinuousLagrangeSpace(grid, order)
    op = H.make_matrix_operator(space, H.Stencil.element)
    op.append(H.LocalElementIntegralBilinearForm(H.LocalLaplaceIntegrand(kappa)))
    rhs = H.make_vector_functional(space)
    rhs.append(H.LocalElementIntegralFunctional(H.LocalProductIntegrand().with_ansatz(1.0)))
    op.append(rhs)
    op.append(H.make_dirichlet_constraints(space, H.AllDirichletBoundaryInfo()))
    return space, op


@pytest.mark.parametrize("items", [1, 2, 4, 8])
@pytest.mark.parametrize("geometry,order,cells", [("quad", 1, [61, 50]), ("tri", 2, [31, 40]), ("hex", 2, [7, 8, 6])])
def test_general_storage_rows_per_lane(hgdt_mod, geometry, order, cells, items):
    """rows of at most 9, 19 and 125 entries: held in registers or read in every step, by rows per lane"""
    print(f"case sell64 {geometry} order {order} {cells} items {items}", flush=True)
    space, op = _poisson(hgdt_mod, geometry, order, cells, 13)
    op.set_format("sell64")
    op.set_launch(3, 512, items)
    op.set_launch(4, 512, items)
    op.assemble()
    wg = _both(hgdt_mod, op)
    assert wg == -(-space.num_DoFs // (512 * items))


@pytest.mark.parametrize("geometry,order,cells,taken", [
    ("quad", 1, [1, 2], True), ("quad", 1, [31, 15], True), ("quad", 1, [22, 22], True), ("quad", 1, [180, 190], True),
    ("quad", 1, [400, 351], True), ("tri", 2, [40, 33], True), ("tri", 2, [120, 101], True), ("tet", 1, [14, 9, 21], True),
    ("tet", 2, [6, 5, 7], True), ("hex", 2, [9, 8, 7], True), ("tet", 1, [60, 90, 50], True),
    ("quad", 1, [1100, 999], False)])
def test_general_storage(hgdt_mod, geometry, order, cells, taken):
    """SELL storage: halos as row lists (the last: more rows than the CUs hold)"""
    H = hgdt_mod
    print(f"case sell64 {geometry} order {order} {cells}", flush=True)
    space, op = _poisson(H, geometry, order, cells, 9)
    op.set_format("sell64")
    op.assemble()
    wg = _both(H, op)
    print(f"  {space.num_DoFs} DoFs, {wg} workgroups, {op.last_solve['iterations']} iterations")
    assert (wg > 0) == taken


def test_general_storage_batch_and_scattered_numbering(hgdt_mod):
    """instances of one and of several workgroups, and vertices numbered at random (every workgroup reads most rows)"""
    H = hgdt_mod
    print("case sell64 batch", flush=True)
    parts = [H.Grid.structured("quad", [0, 0], [1, 1], [m, m]) for m in (5, 70, 33, 20)]
    union = H.Grid.union(parts)
    kappa = torch.from_numpy(H.fields.lognormal(7, union.num_elements)).cuda()
    op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=union)[2]
    op.set_format("sell64")
    op.assemble()
    assert _both(H, op) >= 4
    print("case scattered numbering", flush=True)
    g = H.Grid.structured("tri", [0, 0], [1, 1], [70, 60])
    coords, conn = g.coordinates(), g.connectivity()
    perm = np.random.default_rng(3).permutation(len(coords)).astype(np.int32)
    shuffled = np.empty_like(coords)
    shuffled[perm] = coords
    grid = H.Grid.from_arrays("tri", shuffled, perm[conn])
    kappa = torch.from_numpy(H.fields.lognormal(7, grid.num_elements)).cuda()
    op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=grid)[2]
    op.assemble()
    assert _both(H, op) > 1 and op.format_info()["format"] == "sell64"


def test_batch_of_several_rounds(hgdt_mod):
    """more rows than the CUs hold at once: workgroups take one instance after the other, those of an instance together"""
    H = hgdt_mod
    print("case batch of several rounds", flush=True)
    sizes = [380, 11, 250, 31, 380, 300, 90, 380, 2, 380, 380, 199, 380, 45, 380, 380, 380, 64, 380, 380, 380]
    parts = {m: H.Grid.structured("quad", [0, 0], [1, 1], [m, m]) for m in set(sizes)}
    union = H.Grid.union([parts[m] for m in sizes])
    kappa = torch.from_numpy(H.fields.lognormal(7, union.num_elements)).cuda()
    grid, space, op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=union)
    op.assemble()
    wg = _both(H, op)
    print(f"  {space.num_DoFs} DoFs, {wg} workgroups")
    assert 0 < wg <= 256 and space.num_DoFs > 8192 * 200
