"""Equivariant / indexed linear: values vs the oracle's block linear, gradients by gradcheck (CPU, fp64).

The Linear's GEMMs are torch.mm calls that run on whatever device the tensors
are on, so its block bookkeeping and hand-written backward are checked here on
the CPU; on the GPU it is exercised by the MACE parity tests.
"""

import numpy as np
import torch

from molnex_amd.molrep.interaction.linear import Linear
from oracle import mace_ref


def _blocks(s):
    out = []
    for tok in s.split("+"):
        mul, ir = tok.strip().split("x")
        out.append((int(mul), int(ir[:-1]), 1 if ir[-1] == "e" else -1))
    return out


def test_block_linear_matches_oracle_and_gradcheck():
    torch.manual_seed(0)
    ins = "3x0e + 2x1o + 4x0e + 3x1o + 2x2e"
    outs = "5x0e + 2x1o + 3x2e"
    lin = Linear(ins, outs, dtype=torch.float64)
    x = torch.randn(7, lin.irreps_in.dim, dtype=torch.float64, requires_grad=True)
    ref = mace_ref.linear(x.detach(), lin.weight.detach(), _blocks(ins), _blocks(outs))
    np.testing.assert_allclose(lin(x).detach().numpy(), ref.numpy(), atol=1e-12)
    assert torch.autograd.gradcheck(lambda a, w: lin._mix(a, w), (x, lin.weight.detach().reshape(-1).clone()
                                                                    .requires_grad_(True)))


def test_indexed_linear_gradcheck():
    torch.manual_seed(1)
    lin = Linear("6x0e", "6x0e", internal_weights=False, weight_classes=3, dtype=torch.float64)
    x = torch.randn(11, 6, dtype=torch.float64, requires_grad=True)
    W = torch.randn(3, 36, dtype=torch.float64, requires_grad=True)
    z = torch.tensor([0, 2, 2, 1, 0, 0, 2, 1, 1, 0, 2])
    out = lin(x, weight=W, weight_indices=z)
    ref = torch.stack([x[i] @ W[z[i]].view(6, 6) / np.sqrt(6) for i in range(11)])
    np.testing.assert_allclose(out.detach().numpy(), ref.detach().numpy(), atol=1e-12)
    assert torch.autograd.gradcheck(lambda a, w: lin(a, weight=w, weight_indices=z), (x, W))


def test_radial_mlp_chunked_last_layer_matches_dense(monkeypatch):
    """The row-chunked last layer (used for large edge counts) equals the plain layer,
    values and gradients, including a ragged final chunk."""
    import torch.nn.functional as F

    from molnex_amd.molrep.interaction import radial_mlp as R

    monkeypatch.setattr(R, "_CHUNK", 7)
    torch.manual_seed(0)
    x = torch.randn(30, 5, dtype=torch.float64, requires_grad=True)
    W = torch.randn(11, 5, dtype=torch.float64, requires_grad=True)
    b = torch.randn(11, dtype=torch.float64, requires_grad=True)
    g = torch.randn(30, 11, dtype=torch.float64)
    out = R._ChunkedLinear.apply(x, W, b)
    ref = F.linear(x, W, b)
    assert torch.allclose(out, ref, atol=1e-12)
    got = torch.autograd.grad(out, (x, W, b), g)
    exp = torch.autograd.grad(ref, (x, W, b), g)
    for a, e in zip(got, exp):
        assert torch.allclose(a, e, atol=1e-12)


def test_linear_input_irrep_without_output_gets_zero_grad():
    from molnex_amd.molrep.interaction import Linear

    torch.manual_seed(1)
    lin = Linear("4x0e+3x1o+2x2e", "5x0e+2x2e", dtype=torch.float64)
    x = torch.randn(6, 4 + 9 + 10, dtype=torch.float64, requires_grad=True)
    assert torch.autograd.gradcheck(lambda a, w: lin(a, weight=w), (x, lin.weight.detach().clone().requires_grad_()))
    (gx,) = torch.autograd.grad(lin(x).sum(), (x,))
    assert torch.all(gx[:, 4:13] == 0) and gx[:, :4].abs().sum() > 0


def test_polynomial_cutoff_factored_form_matches_expanded_formula():
    """The factored evaluation of the polynomial envelope is the reference's formula
    (src/molrep/embedding/cutoff.py:138-161): equal in fp64 for p = 1..9 over [0, 1.2]; in fp32
    near the cutoff it stays within 1e-7 of the fp64 value where the expanded sum does not."""
    from math import comb

    from molnex_amd.molrep.embedding.cutoff import PolynomialCutoff

    r = torch.linspace(0, 6.0, 4001, dtype=torch.float64)
    for p in range(1, 10):
        x = r / 5.0
        ref = 1 - comb(p + 2, 2) * x ** p + p * (p + 2) * x ** (p + 1) - comb(p + 1, 2) * x ** (p + 2)
        ref = torch.where(x < 1, ref, torch.zeros_like(ref))
        got = PolynomialCutoff(r_cut=5.0, exponent=p)(r.float()).double()
        assert (got - ref).abs().max() < 1e-6, p
    rn = torch.linspace(4.5, 4.99999, 20001)
    xd = rn.double() / 5.0
    exact = 1 - 28 * xd ** 6 + 48 * xd ** 7 - 21 * xd ** 8
    assert (PolynomialCutoff(r_cut=5.0)(rn).double() - exact).abs().max() < 1e-7
    x32 = rn / 5.0
    expanded32 = 1 - 28 * x32 ** 6 + 48 * x32 ** 7 - 21 * x32 ** 8
    assert (expanded32.double() - exact).abs().max() > 1e-6  # the cancellation the factored form avoids


def test_a_module_pickled_with_other_launch_lists_gets_its_own():
    """Launch lists are derived from the irreps when a pickled module is read: one saved before the weights were
    read in place held {"fwd", "bwd"} and fragment tables as buffers."""
    import copy
    import io

    for kw in ({}, {"weight_classes": 3}):
        lin = Linear("8x0e+16x1o", "8x0e+8x1o", **kw)
        plan = lin._hip_plan
        old = copy.deepcopy(lin)
        old._hip_plan = {"fwd": plan["fwd"], "bwd": []}
        for name in ("idx_f", "sc_f", "idx_b", "sc_b"):
            torch.nn.Module.register_buffer(old, "_hip_" + name + "_", torch.zeros(3), persistent=False)
        buf = io.BytesIO()
        torch.save(old, buf)
        buf.seek(0)
        got = torch.load(buf, weights_only=False)
        assert got._hip_plan == plan and not list(got.buffers())
        assert torch.equal(got._hip_idx_f, lin._hip_idx_f) and torch.equal(got._hip_sc_f, lin._hip_sc_f)
        assert got.state_dict().keys() == lin.state_dict().keys()
    assert Linear("3x0e", "3x0e")._hip_plan is None and copy.deepcopy(Linear("3x0e", "3x0e"))._hip_plan is None
