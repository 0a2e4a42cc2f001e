"""The receiver-walked tensor product's launch forms against the float64 oracle: all path groups in one
launch (few receivers), two and four receivers per wavefront (at most 32 / 16 channels), one launch per group
with one channel per lane (at most 64 channels); on both sides of the number of receivers that separates them, with receivers
of no edge and counts that leave a wavefront partly filled."""

import numpy as np
import pytest
import torch

import molnex_amd.kernels as K
from oracle import equivariant as EQ

pytestmark = pytest.mark.gpu
DEV = "cuda"
# fp32 sums of at most a few hundred products per entry
REL = 1e-6


def _irr(ls, mul=None):
    return "+".join((f"{mul}x" if mul else "") + f"{l}{'eo'[l % 2]}" for l in ls)


@pytest.mark.parametrize("ins,shs", [((0, 1, 2), (0, 1, 2)), ((0, 1), (0, 1, 2, 3)), ((0,), (0, 1, 2, 3))])
@pytest.mark.parametrize("C,N", [(8, 1), (8, 301), (16, 4097), (17, 63), (24, 4099), (32, 5001), (40, 700), (48, 3501),
                                 (64, 3500), (64, 4101), (96, 1750), (128, 1751)])
def test_forward_and_gradients(ins, shs, C, N):
    rng = np.random.default_rng(C + N)
    outs = shs
    cfg = K.tp_config_id(list(ins), list(shs), list(outs))
    tp = EQ.ChannelwiseTP(_irr(ins, C), _irr(shs), _irr(outs, C), C)
    # about two edges per receiver: many without any, some with more than four
    E = 2 * N + 3
    ei = np.stack([rng.integers(0, N, E), np.minimum((N * rng.uniform(0, 1, E) ** 1.5).astype(np.int64), N - 1)], 1)
    t = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).to(DEV).requires_grad_(True)  # noqa: E731
    x, Y, w = t(N, tp.nx * C), t(E, sum(2 * l + 1 for l in shs)), t(E, len(tp.paths) * C)
    e = torch.from_numpy(ei).to(DEV)
    out = torch.ops.molix.tp_scatter(x, Y, w, *torch.ops.molix.edge_csr(e, N), cfg, C)
    g = torch.from_numpy(rng.normal(size=tuple(out.shape)).astype(np.float32)).to(DEV)
    got = [out.detach(), *torch.autograd.grad(out, (x, Y, w), g)]
    a = [v.detach().cpu().numpy() for v in (x, Y, w)]
    want = [tp.forward(*a, ei, N), *tp.backward(*a, ei, g.cpu().numpy())]
    for u, v in zip(got, want):
        u = u.cpu().double().numpy()
        assert np.linalg.norm(u - v) <= REL * np.linalg.norm(v)
        assert np.abs(u - v).max() <= 40 * REL * np.abs(v).max()
