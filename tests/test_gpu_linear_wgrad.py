"""Weight gradient of the ir_mul block linear (molix::block_linear_weight_grad) against float64, at the
edges of its 16-row stages, 64-row slabs and 32 / 64-channel tiles, and its own gradients."""

import pytest
import torch

from oracle import mace_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"

# fp32 products with fp32 sums over r rows in random order: the error of a result of r terms is about
# 2^-24 sqrt(r) of the terms' size, its own size sqrt(r) times theirs; 8x for the slowest-converging entries
REL = 8 * 2.0 ** -24


def _blocks(irreps):
    return [(b.mul, b.ir.l, b.ir.p) for b in irreps]


@pytest.mark.parametrize("irr_in,irr_out", [
    ("128x0e+128x1o+128x1o+128x2e", "128x0e+128x1o+128x2e"),  # 64-wide tiles
    ("64x0e+192x3o", "64x0e+64x3o"),
    ("8x0e+24x1o+40x1o", "40x0e+16x1o"),                      # 32-wide tiles, ragged widths
    ("96x2e+32x0e", "200x2e+8x0e"),
])
@pytest.mark.parametrize("rows", [0, 1, 5, 16, 21, 64, 333, 5003])
def test_weight_gradient_vs_float64(irr_in, irr_out, rows):
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(rows + 1)
    lin = Linear(irr_in, irr_out).to(DEV)
    x = torch.randn(rows, lin.irreps_in.dim, device=DEV)
    g = torch.randn(rows, lin.irreps_out.dim, device=DEV)
    (gw,) = torch.autograd.grad(lin(x), lin.weight, g)
    wd = lin.weight.detach().cpu().double().requires_grad_(True)
    ref = mace_ref.linear(x.cpu().double(), wd, _blocks(lin.irreps_in), _blocks(lin.irreps_out))
    (rgw,) = torch.autograd.grad(ref, wd, g.cpu().double())
    assert (gw.cpu().double() - rgw).norm() <= REL * rgw.norm()
    (again,) = torch.autograd.grad(lin(x), lin.weight, g)
    assert torch.equal(gw, again)  # a fixed summation order


def test_many_pairs_strided_rows_and_unaligned_input():
    """More pairs than one launch takes; rows that are a view (a copy is made, the result the same)."""
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(3)
    lin = Linear("+".join(["8x0e"] * 8), "+".join(["8x0e"] * 8)).to(DEV)  # 64 pairs
    wide = torch.randn(201, 65, device=DEV)
    x, g = wide[:, 1:], torch.randn(201, 64, device=DEV)
    (gw,) = torch.autograd.grad(lin(x), lin.weight, g)
    wd = lin.weight.detach().cpu().double().requires_grad_(True)
    ref = mace_ref.linear(x.cpu().double(), wd, _blocks(lin.irreps_in), _blocks(lin.irreps_out))
    (rgw,) = torch.autograd.grad(ref, wd, g.cpu().double())
    assert (gw.cpu().double() - rgw).norm() <= REL * rgw.norm()


def test_gradients_of_the_weight_gradient():
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(4)
    lin = Linear("16x0e+8x1o+8x1o", "24x0e+8x1o").to(DEV)
    x = torch.randn(37, lin.irreps_in.dim, device=DEV, requires_grad=True)
    g = torch.randn(37, lin.irreps_out.dim, device=DEV, requires_grad=True)
    s = torch.randn_like(lin.weight)
    (gw,) = torch.autograd.grad(lin(x), lin.weight, g, create_graph=True)
    got = torch.autograd.grad((gw * s).sum(), (x, g))
    xd, gd = (v.detach().cpu().double().requires_grad_(True) for v in (x, g))
    ref = mace_ref.linear(xd, s.cpu().double(), _blocks(lin.irreps_in), _blocks(lin.irreps_out))
    want = torch.autograd.grad((ref * gd).sum(), (xd, gd))
    for a, b in zip(got, want):
        assert (a.cpu().double() - b).norm() <= 1e-6 * b.norm()


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), 3.4e38, float("nan")])
@pytest.mark.parametrize("irr_in,irr_out", [("64x0e+128x1o", "128x0e+64x1o"), ("8x0e+24x1o", "40x0e+16x1o")])
@pytest.mark.parametrize("rows,at", [(1, 0), (40, 3), (333, 332), (5003, 2600)])
def test_infinite_and_huge_entries(irr_in, irr_out, rows, at, value):
    """Entries that bf16 cannot hold (its largest value is 3.39e38) give what fp32 sums give: infinities of the
    right sign, finite values where the sum is finite, NaN only of 0 * inf, inf - inf or a NaN, and every other
    weight's gradient as without them."""
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(rows)
    lin = Linear(irr_in, irr_out).to(DEV)
    x = torch.randn(rows, lin.irreps_in.dim)
    g = torch.rand(rows, lin.irreps_out.dim) * 0.8 + 0.1  # the sums with 3.4e38 stay finite
    g *= torch.where(torch.rand(g.shape) < 0.5, -1.0, 1.0)
    x[at, 2] = value
    g[at, 1] = 0.0
    if value != 3.4e38:
        g[at, -3] = -value  # a component of the last block: infinities in both operands
    (gw,) = torch.autograd.grad(lin(x.to(DEV)), lin.weight, g.to(DEV))
    wd = lin.weight.detach().cpu().double().requires_grad_(True)
    ref = mace_ref.linear(x.double(), wd, _blocks(lin.irreps_in), _blocks(lin.irreps_out))
    (want,) = torch.autograd.grad(ref, wd, g.double())
    got = gw.cpu().double()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf])
    big = want.abs() > 1e30
    for part in (torch.isfinite(want) & ~big, torch.isfinite(want) & big):
        assert (got[part] - want[part]).norm() <= REL * want[part].norm()
    assert torch.isfinite(want).sum() > 0.5 * want.numel() and (value != 3.4e38 or (torch.isfinite(want) & big).any())
