"""Every block of an ir_mul linear in one launch (molix::block_linear_weights) against float64: row tiles
(32 to 128 rows per workgroup), 32-row weight chunks, column tiles and groups, blocks that share rows,
class-wise weights."""

import pytest
import torch

from molnex_amd import kernels as K
from oracle import mace_ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
# 2^-24 relative rounding of products and sums over at most 1024 terms in random order
REL = 2.0 ** -24 * 32


def _blocks(irreps):
    return [(b.mul, b.ir.l, b.ir.p) for b in irreps]


@pytest.mark.parametrize("irr_in,irr_out", [
    ("8x0e+16x1o+8x1o", "24x0e+8x1o"),                        # one column tile, K below and across a chunk
    ("64x0e+64x1o+64x1o+64x2e", "64x0e+64x1o+64x2e"),         # two column tiles
    ("96x0e+40x1o", "96x0e+72x1o+32x2e"),                     # three tiles, an output block without source
    ("128x0e+128x0e+128x1o+128x1o+128x1o+128x3o", "128x0e+200x1o+128x3o"),  # four tiles, two column groups
    ("+".join(["16x0e"] * 8 + ["8x1o"] * 8 + ["8x2e"] * 8 + ["8x3o"] * 4), "16x0e+8x1o+8x2e+8x3o"),  # > 24 blocks back
])
@pytest.mark.parametrize("rows", [0, 1, 33, 129, 1000, 9001])
def test_linear_vs_float64(irr_in, irr_out, rows):
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(rows)
    lin = Linear(irr_in, irr_out).to(DEV)
    x = torch.randn(rows, lin.irreps_in.dim, device=DEV, requires_grad=True)
    g = torch.randn(rows, lin.irreps_out.dim, device=DEV)
    out = lin(x)
    (gx,) = torch.autograd.grad(out, x, g)
    xd = x.detach().double().cpu().requires_grad_(True)
    w, at, want, start = lin.weight.detach().double().cpu().reshape(-1), 0, [], {}
    for b, o in zip(lin.irreps_in, lin.irreps_in.offsets()):
        start.setdefault(b.ir, []).append((o, b.mul))
    for o in lin.irreps_out:
        srcs = start.get(o.ir, [])
        acc = torch.zeros(rows, o.ir.dim, o.mul, dtype=torch.float64)
        for col, mul in srcs:
            acc = acc + xd[:, col:col + mul * o.ir.dim].reshape(rows, o.ir.dim, mul) @ w[at:at + mul * o.mul].reshape(mul, o.mul)
            at += mul * o.mul
        want.append((acc / max(1, sum(m for _, m in srcs)) ** 0.5).reshape(rows, o.dim))
    ref = torch.cat(want, 1)
    (rgx,) = torch.autograd.grad(ref, xd, g.double().cpu())
    assert (out.detach().double().cpu() - ref.detach()).norm() <= REL * ref.detach().norm()
    assert (gx.double().cpu() - rgx).norm() <= REL * rgx.norm()


@pytest.mark.parametrize("mul,rows", [(8, 70), (64, 300), (128, 1500)])
def test_indexed_linear_vs_per_class(mul, rows):
    """One weight set per class: the rows of each class equal the plain linear with its weights (bit for
    bit: the same products in the same order); rows of an out-of-range class are zero."""
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(mul)
    irr = f"{mul}x0e+{mul}x1o"
    lin, plain = Linear(irr, irr, internal_weights=False, weight_classes=5).to(DEV), Linear(irr, irr).to(DEV)
    w = torch.randn(5, lin.weight_numel, device=DEV)
    z = torch.randint(0, 6, (rows,), device=DEV)  # 5: out of range
    z[z == 3] = 1                                 # an empty class
    x = torch.randn(rows, lin.irreps_in.dim, device=DEV, requires_grad=True)
    g = torch.randn_like(x)
    groups = K.class_groups(z, 5)
    out = torch.ops.molix.block_linear_weights(x, w, *lin._hip_plan["rows"], lin.irreps_out.dim, False, *groups)
    gx = torch.ops.molix.block_linear_weights(g, w, *lin._hip_plan["cols"], lin.irreps_in.dim, True, *groups)
    for c in range(6):
        sel = z == c
        if c == 5:
            assert not out[sel].any() and not gx[sel].any()
            continue
        want = plain(x, weight=w[c:c + 1])
        (wgx,) = torch.autograd.grad(want, x, g)
        assert torch.equal(out[sel], want.detach()[sel]) and torch.equal(gx[sel], wgx[sel])


def test_input_with_infinities_and_bad_arguments():
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(0)
    lin = Linear("40x0e", "8x0e").to(DEV)  # K = 40: the last chunk is mostly padding
    x = torch.randn(40, 40, device=DEV)
    x[7, 39] = float("inf")
    with torch.no_grad():
        out = lin(x)
    assert torch.isfinite(out[torch.arange(40, device=DEV) != 7]).all() and not torch.isfinite(out[7]).any()
    rows, sc = lin._hip_plan["rows"]
    w = lin.weight.detach().reshape(-1)
    for bad in (dict(out_dim=16), dict(a=x[:, :32]), dict(weight=w[:-1]), dict(scales=sc + [1.0])):
        args = dict(a=x, weight=w, blocks=rows, scales=sc, out_dim=8, transposed=False)
        with pytest.raises(ValueError):
            torch.ops.molix.block_linear_weights(*{**args, **bad}.values())


@pytest.mark.parametrize("irr_in,irr_out", [
    ("8x0e+16x1o+8x1o", "24x0e+8x1o"),
    ("96x0e+40x1o", "96x0e+72x1o+32x2e"),                     # three tiles, an output block without source
    ("128x0e+128x0e+128x1o+128x1o+128x1o+128x3o", "128x0e+200x1o+128x3o"),
])
@pytest.mark.parametrize("rows", [0, 1, 129, 1000])
def test_fragment_ordered_weights(irr_in, irr_out, rows):
    """molix::block_linear and molix::indexed_block_linear (weights put into operand order by the caller) give
    the bits of the form that reads the parameter: the same products in the same order.  The classes hold no,
    one and many rows, and some rows are of none."""
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(rows)
    lin = Linear(irr_in, irr_out).to(DEV)
    x = torch.randn(rows, lin.irreps_in.dim, device=DEV)
    idx, sc, fwd, dim = lin._hip_idx_f, lin._hip_sc_f, lin._hip_plan["fwd"], lin.irreps_out.dim
    with torch.no_grad():
        w = lin.weight.reshape(-1)
        assert torch.equal(torch.ops.molix.block_linear(x, w[idx] * sc, fwd, dim), lin(x))
    if rows == 0:  # the indexed forms take at least one row
        return
    ws = torch.randn(4, lin.weight_numel, device=DEV)
    z = torch.randint(0, 3, (rows,), device=DEV) * 2  # 0, 2, 4: classes 1 and 3 are empty, 4 is none
    if rows > 100:
        z[17] = 3
        z[5] = -1
    groups = K.class_groups(z, 4)
    got = torch.ops.molix.indexed_block_linear(x, ws[:, idx] * sc, *groups, fwd, dim)
    want = torch.ops.molix.block_linear_weights(x, ws, *lin._hip_plan["rows"], dim, False, *groups)
    assert torch.equal(got, want) and not got[(z < 0) | (z > 3)].any()
    per_class = torch.cat([lin(x[n:n + 1], weight=ws[c:c + 1]) if 0 <= c < 4 else torch.zeros(1, dim, device=DEV)
                           for n, c in enumerate(z.tolist()[:40])])
    assert torch.equal(got[:40], per_class)
