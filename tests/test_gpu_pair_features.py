"""The two-body input rows of an edge model (molix::pair_features: radial features, both atoms' type
embeddings and the cutoff envelope in one kernel) against the float64 formulas: row lengths with and
without 16-byte pieces, edge counts around a workgroup's 64, first and second derivatives.

Tolerances: 1e-5 relative to the reference's RMS, as for the radial features alone; the embedding
columns are copies and exact.
"""

import pytest
import torch

import molnex_amd.kernels as K
import molnex_amd.second_order as S

pytestmark = pytest.mark.gpu
DEV = "cuda"
RC = 5.0


def _close(a, b):
    a, b = a.detach().double().cpu(), b.detach().double()
    scale = b.pow(2).mean().sqrt().clamp(min=1e-30)
    assert ((a - b).abs().max() / scale) <= 1e-5


@pytest.mark.parametrize("E,nb,dim,cutoff,norm", [(1, 8, 16, 2, True), (63, 8, 16, 2, True), (64, 4, 4, 1, False),
                                                  (65, 5, 3, 2, True), (1000, 32, 16, 1, True),
                                                  (1000, 8, 7, 2, False), (4097, 8, 0, 2, True),
                                                  (4097, 1, 16, 0, False)])
def test_pair_features_vs_fp64(E, nb, dim, cutoff, norm):
    g = torch.Generator().manual_seed(E + nb)
    r64 = (0.1 + torch.rand(E, dtype=torch.float64, generator=g) * RC * 1.1).float().double().requires_grad_(True)
    ti, tj = (torch.randint(0, 9, (E,), generator=g) for _ in range(2))
    table = torch.randn(9, dim, generator=g)
    mu = torch.randn(nb, generator=g) * 0.1 if norm else None
    sg = 0.5 + torch.rand(nb, generator=g) if norm else None
    rad = S.bessel_cutoff_torch(r64, nb, RC, 1e-8, mu, sg, cutoff, 6)
    u64 = S.envelope_torch(r64, RC, cutoff, 6)
    gf, gu = torch.randn(E, nb + 2 * dim, generator=g), torch.randn(E, generator=g)
    total = (rad * gf[:, :nb].double()).sum() + (u64 * gu.double()).sum()
    (gr64,) = torch.autograd.grad(total, r64, create_graph=True)
    v = torch.randn(E, generator=g)
    second = torch.autograd.grad((gr64 * v.double()).sum(), r64)[0]

    cu = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    r = r64.detach().float().to(DEV).requires_grad_(True)
    out, u = K.pair_features(r, cu(ti), cu(tj), cu(table), nb, RC, 1e-8, cu(mu), cu(sg), cutoff, 6)
    assert out.shape == (E, nb + 2 * dim) and u.shape == (E,)
    assert torch.equal(out[:, nb:].cpu(), torch.cat([table[ti], table[tj]], 1))
    _close(out[:, :nb], rad)
    _close(u, u64)
    (gr,) = torch.autograd.grad((out * cu(gf)).sum() + (u * cu(gu)).sum(), r, create_graph=True)
    _close(gr, gr64)
    _close(torch.autograd.grad((gr * cu(v)).sum(), r)[0], second)


def test_type_outside_the_table_and_no_edges():
    table = torch.randn(3, 4, device=DEV)
    t = torch.tensor([0, 3, -1, 2], device=DEV)
    out, u = K.pair_features(torch.ones(4, device=DEV), t, t.flip(0), table, 4, RC, 1e-8, None, None, 2, 6)
    nan = torch.isnan(out).cpu()
    assert not nan[:, :4].any() and not torch.isnan(u).any()
    assert nan[:, 4].tolist() == [False, True, True, False] and nan[:, 8].tolist() == [False, True, True, False]
    e = torch.empty(0, dtype=torch.int64, device=DEV)
    out, u = K.pair_features(torch.empty(0, device=DEV), e, e, table, 4, RC, 1e-8, None, None, 2, 6)
    assert out.shape == (0, 12) and u.shape == (0,)


@pytest.mark.parametrize("kind", ["forward", "pre", "backward", "global", "own"])
def test_hooks_of_the_basis_and_the_cutoff_run(kind):
    """The embedding calls its modules where a hook (or a forward of the instance's own) waits on them."""
    from molnex_amd.molzoo.allegro import PairEmbedding

    torch.manual_seed(0)
    emb = PairEmbedding(num_elements=4, num_scalar_features=16, num_tensor_features=16, r_max=RC, l_max=1).to(DEV)
    for p in emb.parameters():
        p.requires_grad_(False)
    mods = (emb.radial_basis, emb.cutoff_fn)
    ei, d = torch.randint(0, 10, (70, 2), device=DEV), torch.randn(70, 3, device=DEV)
    z, r = torch.randint(0, 4, (10,), device=DEV), d.norm(dim=-1).requires_grad_(True)
    plain = emb(z, r, d, ei)
    seen = []

    def note(m, *_):
        if m in mods:
            seen.append(m)

    handles = []
    if kind == "global":
        handles.append(torch.nn.modules.module.register_module_forward_hook(note))
    for m in mods:
        if kind == "forward":
            handles.append(m.register_forward_hook(note))
        elif kind == "pre":
            handles.append(m.register_forward_pre_hook(note))
        elif kind == "backward":
            handles.append(m.register_full_backward_hook(note))
        elif kind == "own":
            m.forward = lambda r, m=m, f=m.forward: (note(m), f(r))[1]
    try:
        out = emb(z, r, d, ei)
        torch.autograd.grad(sum(t.sum() for t in out), r)
    finally:
        for h in handles:
            h.remove()
    assert set(seen) == set(mods)
    for a, b in zip(out, plain):
        _close(a, b.cpu())
