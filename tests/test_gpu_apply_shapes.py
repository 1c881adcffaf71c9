"""Operator applications over row blocks of several rows per lane: split over workgroups of 256 lanes, of the block's own
lanes where 256 do not divide its rows, remainders at the end of an instance and instances smaller than a workgroup.  A
row's sum does not depend on the blocks: the bits of one row per lane."""
import pytest
import torch

from problems import hgdt_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["auto", "dia", "sell64"])
@pytest.mark.parametrize("sizes", [[1], [15, 16], [2, 90, 3, 61, 33]])
def test_products_of_all_shapes(hgdt_mod, fmt, sizes):
    H = hgdt_mod
    print(f"case {fmt} {sizes}", flush=True)
    parts = [H.Grid.structured("quad", [0, 0], [1, 1], [m, m + 1]) for m in sizes]
    grid = H.Grid.union(parts) if len(parts) > 1 else parts[0]
    kappa = torch.from_numpy(H.fields.lognormal(7, grid.num_elements)).cuda()
    space, op = hgdt_problem(H, "heat_q1", None, kappa, grid=grid)[1:]
    op.set_format(fmt)
    op.assemble()
    x = torch.from_numpy(H.fields.uniform(8, space.num_DoFs)).cuda()
    op.set_launch(3, 256, 1)
    want = op.apply(x)
    assert torch.isfinite(want).all() and torch.count_nonzero(want) > 0
    for shape in ((64, 1), (64, 2), (64, 4), (192, 2), (192, 4), (320, 4), (512, 4), (768, 4), (512, 8), (1024, 16)):
        print(f"  {shape}", flush=True)
        op.set_launch(3, *shape)
        got = op.apply(x, torch.full_like(want, float("nan")))
        assert torch.equal(got, want), shape
