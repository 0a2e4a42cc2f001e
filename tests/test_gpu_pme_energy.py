"""molix::pme_energy (the whole PME term in one op) against the ops it stands for: the neighbor list's pairs
through molix::pme_direct, molix::pme_reciprocal and the self term, in float64, over the paths of its pair
scan (all pairs, cells, crowded cells, all-pairs grids) and the mesh kernels' orders and edges."""

import math

import pytest
import torch

import molnex_amd.kernels  # noqa: F401
from molnex_amd.molpot import PMEPotential

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _composed(pme, pos, q, box):
    """The module's form for given pairs, in float64."""
    pos, q, box = (t.detach().double() for t in (pos, q, box))
    pos.requires_grad_(True), q.requires_grad_(True)
    i, j, _, d, r = torch.ops.molix.neighbor_list(pos.detach(), pme.cutoff, box, False)
    e = pme(pos, q, box, pairs=(torch.stack([i, j]), d, r))
    gp, gq = torch.autograd.grad(e, (pos, q))
    return e.detach(), gp, gq


def _run(pme, pos, q, box):
    p, c = pos.clone().requires_grad_(True), q.clone().requires_grad_(True)
    e = pme(p, c, box)
    gp, gq = torch.autograd.grad(e, (p, c))
    return e.detach(), gp, gq


def _close(got, want, tol, terms=0.0):
    """``terms``: the size of the terms a result is the difference of.  The mesh force of an atom on itself,
    for one, is order^3 terms of size k q^2 alpha that cancel to the spline's error; their rounding stays."""
    for a, b in zip(got, want):
        assert a.shape == b.shape
        bound = tol * b.norm().item() + torch.finfo(a.dtype).eps / 2 * terms
        assert (a.double() - b).norm() <= bound, ((a.double() - b).norm(), b.norm())


def _system(n, edge, seed, box=None):
    g = torch.Generator().manual_seed(seed)
    box = torch.eye(3, dtype=torch.float64) * edge if box is None else box
    k = math.ceil(n ** (1 / 3))
    grid = torch.stack(torch.meshgrid(*[torch.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)
    sites = grid[torch.randperm(k ** 3, generator=g)[:n]].double()
    # jittered lattice: pairs stay apart, so no single 1/r term decides the result
    pos = ((sites + 0.25 + 0.5 * torch.rand(n, 3, generator=g, dtype=torch.float64)) / k) @ box
    q = torch.randn(n, generator=g, dtype=torch.float64)
    return pos.to(DEV), (q - q.mean() if n > 1 else q).to(DEV), box.to(DEV)


# float64: both sides sum the same terms in other orders.  float32: positions and charges are rounded
# identically for both sides (the oracle gets the rounded values); mesh sums of ~order^3 terms at 2^-24.
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-11), (torch.float32, 2e-5)])
@pytest.mark.parametrize("n,edge,cut,mesh,order,kind", [
    (1, 9.0, 3.0, (16, 16, 16), 4, "cubic"),
    (2, 9.0, 4.0, (12, 16, 20), 5, "cubic"),
    (130, 11.0, 5.0, (16, 17, 18), 6, "cubic"),         # under three cutoffs: exact images only
    (700, 19.0, 5.0, (9, 11, 8), 8, "cubic"),           # a mesh of one brick and a bit
    (2047, 27.0, 4.0, (24, 24, 24), 3, "cubic"),
    (2049, 27.0, 4.0, (26, 30, 28), 7, "triclinic"),    # the cell scan
    (4000, 22.0, 5.0, (32, 32, 32), 4, "cubic"),        # about 200 neighbours
    (3000, 30.0, 4.0, (16, 64, 16), 5, "thin"),         # two cells along one axis: an all-pairs grid
])
def test_energy_and_gradients(n, edge, cut, mesh, order, kind, dtype, tol):
    box = None
    if kind == "triclinic":
        box = torch.tensor([[edge, 0, 0], [0.2 * edge, edge, 0], [-0.1 * edge, 0.3 * edge, edge]], dtype=torch.float64)
    if kind == "thin":
        box = torch.diag(torch.tensor([edge, 3 * edge, 9.0], dtype=torch.float64))
    pos, q, box = (t.to(dtype) for t in _system(n, edge, n + order, box))
    pme = PMEPotential(alpha=0.4, grid=mesh, order=order, cutoff=cut).to(DEV)
    want = _composed(pme, pos, q, box)
    got = _run(pme, pos, q, box)
    _close(got, want, tol, pme.coulomb * pme.alpha * float((q.double() ** 2).sum()))
    # bitwise the same again (the cell scan: test_the_same_bits_every_time)
    again = _run(pme, pos, q, box)
    if n <= 2048:
        assert all(torch.equal(a, b) for a, b in zip(got, again))
    else:
        _close(again, [t.double() for t in got], tol)


@pytest.mark.parametrize("n,edge,cut", [(2049, 27.0, 4.0), (9000, 45.0, 5.0), (6000, 45.0, 14.9)])
def test_the_same_bits_every_time(n, edge, cut):
    """The cell scan sums in a fixed order: energy and gradients are reproducible in float64.  (The last size has
    27 cells of 220 atoms.)"""
    pos, q, box = _system(n, edge, 11)
    pme = PMEPotential(alpha=0.4, grid=(32, 32, 32), order=4, cutoff=cut).to(DEV)
    first = _run(pme, pos, q, box)
    for _ in range(7):
        assert all(torch.equal(a, b) for a, b in zip(_run(pme, pos, q, box), first))


def test_single_gradients_scaling_and_no_grad():
    pos, q, box = (t.float() for t in _system(600, 18.0, 1))
    pme = PMEPotential(alpha=0.35, grid=(20, 20, 20), order=5, cutoff=4.5).to(DEV)
    e, gp, gq = _run(pme, pos, q, box)
    with torch.no_grad():
        assert torch.equal(pme(pos, q, box), e)
    p = pos.clone().requires_grad_(True)
    (only,) = torch.autograd.grad(3.0 * pme(p, q, box), p)
    torch.testing.assert_close(only, 3.0 * gp, rtol=1e-6, atol=1e-6)
    c = q.clone().requires_grad_(True)
    (only,) = torch.autograd.grad(pme(pos, c, box), c)
    torch.testing.assert_close(only, gq, rtol=1e-6, atol=1e-6)
    # the forward told that no gradient is wanted: the backward forms the real-space part itself
    spec = torch.ops.molix.pme_energy(pos, q, box, pme.xmoduli, pme.ymoduli, pme.zmoduli, 20, 20, 20, 5, 0.35, 4.5, pme.coulomb, False)
    got = torch.ops.molix.pme_energy_backward(torch.ones((), device=DEV), pos, q, box, *spec[1:], 20, 20, 20, 5, 0.35, 4.5,
                                              pme.coulomb)
    assert torch.equal(got[0], gp) and torch.equal(got[1], gq)


@pytest.mark.parametrize("n", [1, 600])
@pytest.mark.parametrize("shape", [(-1, 1), (1, -1)])
def test_charges_in_a_column_or_a_row(n, shape):
    pos, q, box = _system(n, 18.0, 1)
    pme = PMEPotential(alpha=0.35, grid=(20, 20, 20), order=5, cutoff=4.5).to(DEV)
    e, gp, gq = _run(pme, pos, q, box)
    got = _run(pme, pos, q.reshape(shape), box)
    assert torch.equal(got[0], e) and torch.equal(got[1], gp) and torch.equal(got[2], gq.reshape(shape))
    with pytest.raises((ValueError, RuntimeError)):
        pme(pos, torch.zeros(n + 1, device=DEV, dtype=pos.dtype), box)


def test_too_many_neighbours_is_refused():
    pos = torch.rand(4300, 3, device=DEV) * 2.0
    pme = PMEPotential(alpha=0.3, grid=(16, 16, 16), order=4, cutoff=4.0).to(DEV)
    with pytest.raises(RuntimeError, match="4096"):
        pme(pos, torch.zeros(4300, device=DEV), torch.eye(3, device=DEV) * 20.0)


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-11), (torch.float32, 2e-5)])
@pytest.mark.parametrize("box", [(30.0, 12.0, 12.0), (30.0, 8.0, 8.0)])  # the cell scan, an all-pairs grid
def test_dense_sorted_systems_within_the_half_lists_limit(box, dtype, tol):
    """Up to 6000 neighbours an atom, at most 3000 of lower index: the limit of 4096 is the half list's, so such
    a system is taken (tolerances as above)."""
    n, g = 12000, torch.Generator().manual_seed(1)
    pos = 1.0 + 0.5 * torch.rand(n, 3, generator=g, dtype=torch.float64)
    pos[:, 0] = 0.001 * torch.arange(n)
    q = torch.randn(n, generator=g, dtype=torch.float64)
    pos, q, box = (t.to(DEV, dtype) for t in (pos, q - q.mean(), torch.diag(torch.tensor(box, dtype=torch.float64))))
    pme = PMEPotential(alpha=0.4, grid=(32, 32, 32), order=4, cutoff=3.0).to(DEV)
    want = _composed(pme, pos, q, box)
    _close(_run(pme, pos, q, box), want, tol, pme.coulomb * pme.alpha * float((q.double() ** 2).sum()))


def test_the_neighbour_flag_is_awaited_on_the_tensors_stream(monkeypatch):
    """The flag's event is recorded on the stream of the positions' device, which need not be the current one."""
    seen = []

    class Event(torch.cuda.Event):
        def record(self, stream=None):
            seen.append(stream)
            super().record(torch.cuda.current_stream() if stream is None else stream)

    monkeypatch.setattr(torch.cuda, "Event", Event)
    pos, q, box = _system(4200, 35.0, 2)
    pme = PMEPotential(alpha=0.4, grid=(32, 32, 32), order=4, cutoff=4.0).to(DEV)
    side = torch.cuda.Stream(pos.device)
    side.wait_stream(torch.cuda.current_stream(pos.device))
    with torch.cuda.stream(side):
        pme(pos, q, box)
    torch.cuda.synchronize()
    assert seen == [side]


@pytest.mark.parametrize("sfx", ["f32", "f64"])
@pytest.mark.parametrize("n", [1, 100, 2047, 2048, 2049, 5003])
def test_the_neighbour_flag_and_the_workspace(n, sfx):
    """The flag is always written, and nothing behind the workspace that was asked for."""
    from molnex_amd import _lib

    lib, ptr = _lib.load(), _lib.ptr
    pos, q, box = (t.to(torch.float32 if sfx == "f32" else torch.float64) for t in _system(n, 28.0, 3))
    parts = torch.zeros(lib.mnx_pme_real_partials(n), dtype=torch.float64, device=DEV)
    flag = torch.full((1,), -1, dtype=torch.int32, device=DEV)
    need = lib.mnx_pme_real_workspace_bytes(n, sfx == "f64")
    ws = torch.full((need + 65536,), 0x5a, dtype=torch.uint8, device=DEV)
    dpos, dq = torch.empty_like(pos), torch.empty_like(q)
    _lib.check(getattr(lib, f"mnx_pme_real_{sfx}")(
        ptr(pos), ptr(q), n, ptr(box), 4.0, 0.4, 1.0, ptr(dpos), ptr(dq), ptr(parts), ptr(flag), ptr(ws), need,
        torch.cuda.current_stream().cuda_stream), "real")
    assert flag.item() == 0 and (ws[need:] == 0x5a).all()
    assert torch.isfinite(dpos).all() and torch.isfinite(dq).all()


@pytest.mark.parametrize("n", [1500, 4097])
def test_captured_graph_replays(n):
    """Systems whose atoms cannot exceed the neighbour limit read nothing back, so a graph can hold the term: every
    replay equals the eager result, with eager work in between."""
    pos, q, box = (t.float() for t in _system(n, (n / 0.1) ** (1 / 3), 4))
    pme = PMEPotential(alpha=0.4, grid=(32, 32, 32), order=4, cutoff=4.0).to(DEV)
    p = pos.clone().requires_grad_(True)

    def step():
        e = pme(p, q, box)
        return e.detach(), torch.autograd.grad(e, p)[0]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for k in range(5):
        with torch.no_grad():
            p.copy_(pos + 0.1 * k)
        want = [t.clone() for t in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
        torch.randn(500, 500, device=DEV).sum().item()


def test_opcheck():
    pos, q, box = _system(150, 12.0, 5)
    pme = PMEPotential(alpha=0.4, grid=(16, 16, 16), order=4, cutoff=3.5).to(DEV)
    pos.requires_grad_(True), q.requires_grad_(True)
    torch.library.opcheck(torch.ops.molix.pme_energy.default,
                          (pos, q, box, pme.xmoduli, pme.ymoduli, pme.zmoduli, 16, 16, 16, 4, 0.4, 3.5, 1.0, True))


def test_scaled_forces_differentiated_by_the_scale():
    """The gradient is linear in its upstream gradient, also under create_graph: |w F|^2 by w."""
    pos, q, box = _system(300, 15.0, 3)
    pme = PMEPotential(alpha=0.4, grid=(16, 16, 16), order=4, cutoff=4.5).to(DEV)
    _, gp, gq = _run(pme, pos, q, box)
    w = torch.tensor(1.5, dtype=pos.dtype, device=DEV, requires_grad=True)
    p, c = pos.clone().requires_grad_(True), q.clone().requires_grad_(True)
    fp, fq = torch.autograd.grad(w * pme(p, c, box), (p, c), create_graph=True)
    (gw,) = torch.autograd.grad(fp.square().sum() + fq.square().sum(), w, retain_graph=True)
    torch.testing.assert_close(gw, 2 * 1.5 * (gp.square().sum() + gq.square().sum()), rtol=1e-11, atol=0.0)
    with pytest.raises(RuntimeError, match="no autograd formula"):
        torch.autograd.grad(fp.square().sum(), p)
