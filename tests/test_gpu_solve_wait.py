"""Solves whose launch gives up because a wait outlasts its limit (limit 0: a workgroup that the others wait for is left
out; every workgroup then ends through its normal return): the solve starts over with kernels per iteration, from an untouched iterate, residual and
records, so that it has the bits of a timed solve, which takes these kernels anyway.  And solves that wait for CUs which
other solves of the process hold."""
import threading

import numpy as np
import pytest
import torch

from problems import hgdt_problem
from test_gpu_resident import _poisson, _swipdg

pytestmark = pytest.mark.gpu


def _operator(H, case):
    """operators whose solve takes several workgroups"""
    if case == "dia":
        kappa = torch.from_numpy(H.fields.lognormal(7, 150 * 131)).cuda()
        op = hgdt_problem(H, "heat_q1", [150, 131], kappa)[2]
        op.assemble()
    elif case == "far":
        kappa = torch.from_numpy(H.fields.lognormal(7, 86 * 87 * 88 * 6)).cuda()
        op = hgdt_problem(H, "p1_tets", [86, 87, 88], kappa)[2]
        op.assemble()
    elif case in ("hex", "sell"):
        op = _poisson(H, "hex", 1, [30, 31, 29], 13)[1] if case == "hex" else _poisson(H, "tri", 2, [70, 61], 13)[1]
        op.assemble()
    elif case in ("dia batch", "sell batch"):
        grid = H.Grid.union([H.Grid.structured("quad", [0, 0], [1, 1], [m, m]) for m in (3, 150, 22, 64, 97)])
        kappa = torch.from_numpy(H.fields.lognormal(7, grid.num_elements)).cuda()
        op = hgdt_problem(H, "heat_q1", None, kappa, f=1.0, grid=grid)[2]
        op.set_format("sell64" if case == "sell batch" else "auto")
        op.assemble()
    else:
        fmt, batch = case.split(" ")[0], case.endswith("batch")
        parts = [H.Grid.structured("quad", [0, 0], [1, 1], [m, m + 1]) for m in ((3, 60, 23, 41) if batch else (60,))]
        grid = H.Grid.union(parts) if batch else parts[0]
        kappa = torch.from_numpy(H.fields.lognormal(23, grid.num_elements)).cuda()
        op = _swipdg(H, grid, kappa, fmt="auto" if fmt == "blocks" else fmt)[1]
    return op


@pytest.mark.parametrize("case", ["dia", "dia batch", "far", "hex", "sell", "sell batch", "blocks", "blocks batch",
                                  "matrix_free", "matrix_free batch"])
def test_solve_whose_launch_gives_up(hgdt_mod, case):
    H = hgdt_mod
    print(f"case {case}", flush=True)
    op = _operator(H, case)
    n = op.rhs.numel()
    guess = torch.from_numpy(H.fields.uniform(8, n)).cuda()
    opts = [{"precision": 1e-6}, {"precision": 1e-6, "initial_guess": True}]
    alone = op.apply_inverse("rhs", opts=opts[0])
    assert op.solve_workgroups() > 1
    for o in opts:
        print(f"  {o}", flush=True)
        want = op.apply_inverse("rhs", guess.clone(), opts=o, time_spmv=8)
        s2, i2 = dict(op.last_solve), op.instance_stats()
        op.set_solve_wait(0.)
        left, got = 16 if o is opts[1] else 0, None
        while left >= 0:  # (the solves that skip the launch after one that gave up have the same bits)
            got = op.apply_inverse("rhs", guess.clone(), opts=o)
            s1, i1 = dict(op.last_solve), op.instance_stats()
            assert op.solve_workgroups() == 0 and torch.equal(got, want), left
            assert np.array_equal(i1[0], i2[0]) and np.array_equal(i1[1], i2[1])
            for k in ("iterations", "relres", "true_relres", "converged"):
                assert s1[k] == s2[k], k
            left -= 1
        op.set_solve_wait(4.)
    # the second guess's first 16 solves counted down what the first one's left; its last one gave up again
    for k in range(16):
        op.apply_inverse("rhs", guess.clone(), opts={"precision": 0.5})
        assert op.solve_workgroups() == 0, k
    again = op.apply_inverse("rhs", opts=opts[0])
    assert op.solve_workgroups() > 1 and torch.equal(again, alone)


def test_graph_and_limit_of_steps_after_giving_up(hgdt_mod):
    H = hgdt_mod
    print("case graph, stop at max_iter", flush=True)
    op = _operator(H, "dia batch")
    n = op.rhs.numel()
    want = op.apply_inverse("rhs", time_spmv=8)
    op.set_solve_wait(0.)
    assert torch.equal(op.apply_inverse("rhs", use_graph=True, check_every=8), want) and op.solve_workgroups() == 0
    xs = []
    for spmv, wait in ((8, 4.), (0, 0.)):
        fresh = _operator(H, "dia batch")
        fresh.set_solve_wait(wait)
        x = torch.zeros(n, dtype=torch.float64, device="cuda")
        with pytest.raises(H.linear_solver_failed):
            fresh.apply_inverse("rhs", x, opts={"max_iter": 7}, time_spmv=spmv)
        assert fresh.last_solve["iterations"] == 7 and fresh.solve_workgroups() == 0
        xs.append(x)
    assert torch.equal(*xs)


def test_one_workgroup_never_waits(hgdt_mod):
    print("case one workgroup", flush=True)
    kappa = torch.from_numpy(hgdt_mod.fields.lognormal(7, 22 * 22)).cuda()
    op = hgdt_problem(hgdt_mod, "heat_q1", [22, 22], kappa)[2]
    op.assemble()
    want = op.apply_inverse("rhs")
    op.set_solve_wait(0.)
    assert torch.equal(op.apply_inverse("rhs"), want) and op.solve_workgroups() == 1


def test_refused_waits(hgdt_mod):
    kappa = torch.ones(4, dtype=torch.float64, device="cuda")
    op = hgdt_problem(hgdt_mod, "heat_q1", [2, 2], kappa)[2]
    for seconds in (-1., float("nan"), float("inf")):
        with pytest.raises(Exception):
            op.set_solve_wait(seconds)


def test_solves_that_exceed_the_cus_together(hgdt_mod):
    """each takes more than half of the CUs: the second thread's launch waits until the first one's is over"""
    print("case two threads, more than half of the CUs each", flush=True)
    ops, alone = [], []
    for seed, cells in ((11, [900, 900]), (12, [1000, 800])):
        kappa = torch.from_numpy(hgdt_mod.fields.lognormal(seed, cells[0] * cells[1])).cuda()
        op = hgdt_problem(hgdt_mod, "heat_q1", cells, kappa)[2]
        op.assemble()
        alone.append(op.apply_inverse("rhs", opts={"precision": 1e-3}))
        assert op.solve_workgroups() > torch.cuda.get_device_properties(0).multi_processor_count // 2
        ops.append(op)
    torch.cuda.synchronize()
    got, groups = [[], []], [[], []]

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(4):
                got[k].append(ops[k].apply_inverse("rhs", opts={"precision": 1e-3}))
                groups[k].append(ops[k].solve_workgroups())
        s.synchronize()

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    for k in range(2):
        assert len(got[k]) == 4 and all(torch.equal(x, alone[k]) for x in got[k]) and min(groups[k]) > 0


def test_shortest_wait(hgdt_mod):
    """a limit below the clock's resolution is a limit, not 0: the launch is complete, and waits of some microseconds end
    before the clock is looked at"""
    print("case shortest wait", flush=True)
    op = _operator(hgdt_mod, "dia")
    want = op.apply_inverse("rhs", time_spmv=8)
    op.set_solve_wait(1e-12)
    groups = []
    for _ in range(40):  # (were one to give up all the same, the 17th after it is tried again)
        assert torch.equal(op.apply_inverse("rhs"), want)
        groups.append(op.solve_workgroups())
    assert max(groups) > 1
