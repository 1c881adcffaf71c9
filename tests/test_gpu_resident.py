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


@pytest.mark.parametrize("cells,taken", [
    ([1, 1, 1], True), ([2, 3, 2], True), ([7, 7, 7], True), ([12, 9, 15], True), ([30, 31, 29], True),
    ([55, 60, 61], True), ([61, 59, 120], True), ([96, 96, 20], False)])
def test_thirteen_upper_diagonals(hgdt_mod, cells, taken):
    """Q1 on hexahedra: the matrix read in every step; planes too large for LDS are left to the three kernels"""
    print(f"case hex {cells}", flush=True)
    space, op = _poisson(hgdt_mod, "hex", 1, cells, 13)
    op.assemble()
    assert (_both(hgdt_mod, op) > 0) == taken


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


def _swipdg(H, grid, kappa, omega=None, mass=0.0, faces=True, fmt="auto"):
    omega = kappa if omega is None else omega
    space = H.DiscontinuousLagrangeSpace(grid, 1)
    op = H.make_matrix_operator(space, H.Stencil.element_and_intersection if faces else H.Stencil.element)
    op.append(H.LocalElementIntegralBilinearForm(H.LocalLaplaceIntegrand(kappa)))
    if mass:
        op.append(H.LocalElementIntegralBilinearForm(H.LocalProductIntegrand(mass)))
    if faces:
        op.append(H.LocalCouplingIntersectionIntegralBilinearForm(
            H.LocalLaplaceIPDGInnerCoupling(1.0, kappa, omega) + H.LocalIPDGInnerPenalty(16.0, omega)), {},
            H.ApplyOn.InnerIntersectionsOnce())
        op.append(H.LocalIntersectionIntegralBilinearForm(
            H.LocalIPDGBoundaryPenalty(16.0, omega) + H.LocalLaplaceIPDGDirichletCoupling(1.0, kappa)), {},
            H.ApplyOn.CustomBoundaryIntersections(H.AllDirichletBoundaryInfo()))
    rhs = H.make_vector_functional(space)
    rhs.append(H.LocalElementIntegralFunctional(H.LocalProductIntegrand().with_ansatz(1.0)))
    op.append(rhs)
    op.set_format(fmt)
    op.assemble()
    return space, op


def _same_steps(H, space, op, limits=(1, 2, 3, 8)):
    """the iterates of both ways after a few steps: the same sums in another order, so that alpha and beta differ by the
    round-off of sums of up to a million terms (1e-13) and the iterate by a small multiple: bound 1e-11"""
    wg = None
    for limit in limits:
        xs = []
        for spmv in (0, 8):
            x = torch.zeros(space.num_DoFs, dtype=torch.float64, device="cuda")
            try:
                op.apply_inverse("rhs", x, opts={"max_iter": limit}, time_spmv=spmv)
            except H.linear_solver_failed:
                assert op.last_solve["iterations"] == limit
            wg = op.solve_workgroups() if spmv == 0 else wg
            xs.append(x)
        assert float((xs[0] - xs[1]).norm()) <= 1e-11 * float(xs[1].norm()), limit
    return wg


@pytest.mark.parametrize("cells,blocks,matrix_free", [
    ([1, 1], 1, 1), ([2, 3], 1, 1), ([32, 16], 1, 1), ([23, 23], 2, 2), ([1, 700], 2, 2), ([700, 1], 2, 2),
    ([33, 65], 5, 5), ([131, 97], None, None), ([256, 192], 96, 96), ([362, 361], 0, None), ([512, 512], 0, 256),
    ([513, 512], 0, 0)])
@pytest.mark.parametrize("fmt", ["auto", "matrix_free"])
def test_discontinuous_spaces(hgdt_mod, cells, blocks, matrix_free, fmt):
    print(f"case swipdg {fmt} {cells}", flush=True)
    H = hgdt_mod
    grid = H.Grid.structured("quad", [0, 0], [cells[0] / 100, 0.7 * cells[1] / 100], cells)
    kappa = torch.from_numpy(H.fields.lognormal(21, grid.num_elements)).cuda()
    omega = kappa * (1.0 + torch.from_numpy(H.fields.uniform(22, grid.num_elements)).cuda())  # (coercive: a penalty >= kappa's)
    space, op = _swipdg(H, grid, kappa, omega, mass=3.0 if cells[0] % 2 else 0.0, fmt=fmt)
    wg = _same_steps(H, space, op)
    print(f"  {space.num_DoFs} DoFs, {wg} workgroups")
    want = blocks if fmt == "auto" else matrix_free
    assert (wg > 0) if want is None else wg == want
    if space.num_DoFs < 20000:
        x = op.apply_inverse("rhs")
        assert op.last_solve["true_relres"] <= 2e-10
        again = op.apply_inverse("rhs", use_graph=True)
        assert torch.equal(x, again)


@pytest.mark.parametrize("fmt", ["auto", "matrix_free"])
def test_discontinuous_batch(hgdt_mod, fmt):
    """instances of one workgroup and of several, more than fit at once: each with the bits of its own solve (whose first
    residual is summed over the same row blocks)"""
    print(f"case swipdg batch {fmt}", flush=True)
    H = hgdt_mod
    sizes = [3, 40, 1, 150, 64, 23] + [100] * 14
    parts = [H.Grid.structured("quad", [0, 0], [1, 1 + 0.1 * (i % 3)], [m, m + 1]) for i, m in enumerate(sizes)]
    union = H.Grid.union(parts)
    kappa = torch.from_numpy(H.fields.lognormal(23, union.num_elements)).cuda()
    space, op = _swipdg(H, union, kappa, fmt=fmt)
    x = op.apply_inverse("rhs", opts={"precision": 1e-6})
    assert op.solve_workgroups() > 0
    its = op.instance_stats()[0]
    first = np.cumsum([0] + [m * (m + 1) for m in sizes])
    for i in (0, 1, 2, 3, 5, 19):
        s1, op1 = _swipdg(H, parts[i], kappa[int(first[i]):int(first[i + 1])].contiguous(), fmt=fmt)
        for k in (3, 4):
            op1.set_launch(k, *op.get_launch(k))
        x1 = op1.apply_inverse("rhs", opts={"precision": 1e-6})
        assert op1.solve_workgroups() > 0 and op1.last_solve["iterations"] == its[i]
        assert torch.equal(x1, x[4 * int(first[i]):4 * int(first[i + 1])])


def test_element_blocks_of_other_elements(hgdt_mod):
    """simplices (4 neighbours anywhere), an operator without neighbours, and a start from a given iterate"""
    print("case blocks of tets", flush=True)
    H = hgdt_mod
    # (without neighbours the solution is 1: the Laplace part of the product is nothing but round-off, which every step
    # multiplies by its ratio to the mass, so only the first iterate is compared)
    for geometry, cells, faces, limits in (("tet", [7, 6, 5], True, (1, 2, 5)), ("quad", [30, 31], False, (1,))):
        grid = H.Grid.structured(geometry, [0.] * len(cells), [1.] * len(cells), cells)
        kappa = torch.from_numpy(H.fields.lognormal(24, grid.num_elements)).cuda()
        space, op = _swipdg(H, grid, kappa, mass=1.0, faces=faces)
        assert _same_steps(H, space, op, limits) > 0
        guess = torch.from_numpy(H.fields.uniform(8, space.num_DoFs)).cuda()
        got = [op.apply_inverse("rhs", guess.clone(), opts={"initial_guess": True}, time_spmv=spmv) for spmv in (0, 8)]
        assert float((got[0] - got[1]).norm()) <= 1e-8 * float(got[1].norm())
