"""The blocks of a residual linear layer (molix::residual_blocks) against the same float32 products:
each entry is one product (and one sum on the diagonal, which may contract), so 1 ulp of the terms."""

import pytest
import torch

import molnex_amd.kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,F", [(1, 0), (1, 1), (7, 3), (64, 16), (65, 130), (0, 4)])
def test_residual_blocks(S, F):
    g = torch.Generator().manual_seed(S + F)
    wide = torch.randn(S, S + F + 1, generator=g).cuda()
    w, c = wide[:, : S + F], torch.randn(S, generator=g).cuda()
    a, b = 0.8944, 0.4472
    ws, wt, wtt, bc = K.residual_blocks(w, c, a, b)
    eye = torch.eye(S, device="cuda")
    assert torch.equal(wt, w[:, S:] * b) and torch.equal(wtt, (w[:, S:] * b).t()) and torch.equal(bc, c * b)
    ref = eye.double() * a + w[:, :S].double() * b
    assert ((ws.double() - ref).abs() <= 2.0 ** -23 * (eye * a + w[:, :S].abs() * b).double()).all()
