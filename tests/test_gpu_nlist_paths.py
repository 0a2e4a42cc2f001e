"""The neighbor list's paths against the CPU oracle, bit for bit: all-pairs small systems and the cell list
on both sides of the line between them, rows of up to 64, 128, 1024 and more neighbours, all-pairs grids of
more atoms, open and triclinic boxes, both precisions, both lists and both layouts."""

import numpy as np
import pytest
import torch

import molnex_amd.kernels  # noqa: F401
from oracle import nlist as NL

pytestmark = pytest.mark.gpu
DEV = "cuda"
ops = torch.ops.molix


def _same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint8), np.ascontiguousarray(b).view(np.uint8))


def _check(pos, box, cut):
    p = torch.from_numpy(pos).to(DEV)
    b = torch.empty((0, 0), dtype=p.dtype, device=DEV) if box is None else torch.from_numpy(box).to(DEV)
    hi, hj, hd, hr = NL.half_pairs(pos, cut, box)
    i, j, _, d, r = (t.cpu().numpy() for t in ops.neighbor_list(p, cut, b, False))
    assert np.array_equal(i, hi) and np.array_equal(j, hj) and _same(d, hd) and _same(r, hr)
    fi, fj, fd, fr = NL.directed_pairs(pos, cut, box, cells=False)
    i, j, sh, d, r = (t.cpu().numpy() for t in ops.neighbor_list(p, cut, b, True))
    assert np.array_equal(i, fi) and np.array_equal(j, fj) and _same(d, fd) and _same(r, fr)
    for m in (len(hi) // 2, len(hi) + 7) + ((-1,) if len(pos) <= 3000 else ()):
        got = ops.get_neighbor_pairs(p, cut, m, b)
        nb, dd, rr, cnt = NL.get_neighbor_pairs(pos, cut, m if m != len(hi) // 2 else len(hi), box)
        w = got[0].shape[1]
        assert np.array_equal(got[0].cpu().numpy(), nb[:, :w]) and int(got[3]) == len(hi)
        assert _same(np.nan_to_num(got[1].cpu().numpy(), nan=-9), np.nan_to_num(dd[:w], nan=-9))
        assert _same(np.nan_to_num(got[2].cpu().numpy(), nan=-9), np.nan_to_num(rr[:w], nan=-9))
    return np.bincount(fi, minlength=len(pos)).max(initial=0)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 200, 2047, 2048, 2049, 2500])
@pytest.mark.parametrize("kind", ["open", "cubic", "triclinic", "tight"])
def test_sizes_and_boxes(n, kind, dtype):
    """tight: a box of fewer than three cutoffs (half-box distances within the cutoff)."""
    rng = np.random.default_rng(n)
    edge = (n / 0.1) ** (1 / 3)
    box = None if kind == "open" else np.eye(3) * edge
    if kind == "triclinic":
        box = np.array([[edge, 0, 0], [0.2 * edge, edge, 0], [-0.3 * edge, 0.1 * edge, edge]])
    pos = rng.uniform(-0.2, 1.2, (n, 3)) * edge
    cut = 0.49 * edge if kind == "tight" and n <= 200 else min(4.0, 0.3 * edge) if kind != "open" else 4.0
    if kind == "tight" and n > 200:  # three cells along one axis are missing: an all-pairs grid of many atoms
        box = np.diag([edge ** 1.4, edge ** 1.4, edge ** 0.2 * 5])
        pos, cut = rng.uniform(0, 1, (n, 3)) @ box, 3.0
    _check(pos.astype(dtype), None if box is None else box.astype(dtype), cut)


@pytest.mark.parametrize("cut,least,most", [(5.2, 64, 128), (6.5, 128, 1024), (9.0, 300, 1024)])
def test_row_lengths(cut, least, most):
    """More atoms than the all-pairs path takes, neighbour counts around the 64 lanes of one sort, the 128
    entries of a row and beyond."""
    rng = np.random.default_rng(7)
    edge = (6000 / 0.1) ** (1 / 3)
    pos = (rng.uniform(0, 1, (6000, 3)) * edge).astype(np.float32)
    got = _check(pos, (np.eye(3) * edge).astype(np.float32), cut)
    assert least < got <= most
    _check(pos, None, cut)


def test_every_row_length_at_once():
    """A dense cluster in a thin gas: rows of 0 to more than 1024 neighbours, crowded and empty cells."""
    rng = np.random.default_rng(8)
    gas = rng.uniform(0, 90, (3000, 3))
    blob = 45 + rng.normal(size=(1500, 3)) * 1.6
    pos = np.concatenate([gas, blob])[rng.permutation(4500)].astype(np.float32)
    assert _check(pos, (np.eye(3) * 90).astype(np.float32), 4.0) > 1024


@pytest.mark.parametrize("n,full", [(4097, True), (2100, True), (4097, False)])
def test_rows_as_long_as_the_limit(n, full):
    """Every pair of one crowd: rows of up to 4096 neighbours fill the list that a whole workgroup sorts, on the
    cell scan of a wide box and on an all-pairs grid."""
    pos = np.random.default_rng(n).uniform(0, 3, (n, 3)).astype(np.float32)
    p = torch.from_numpy(pos).to(DEV)
    wi, wj = np.nonzero(~np.eye(n, dtype=bool) if full else np.tri(n, k=-1, dtype=bool))
    for edge in (40.0, 14.0):
        i, j, _, d, _ = ops.neighbor_list(p, 6.0, torch.eye(3, device=DEV) * edge, full)
        assert np.array_equal(i.cpu().numpy(), wi) and np.array_equal(j.cpu().numpy(), wj)
        assert torch.equal(d, p[i.long()] - p[j.long()])


def test_duplicates_and_another_stream():
    """Coincident atoms are no pairs (distance 0); a list made on another stream equals the default one's."""
    pos = np.random.default_rng(9).uniform(0, 12, (300, 3)).astype(np.float32)
    pos[10:20] = pos[0:10]
    _check(pos, (np.eye(3) * 14).astype(np.float32), 4.0)
    from molnex_amd.molix.F.locality import neighbor_list

    a = torch.from_numpy(pos).to(DEV)
    s = torch.cuda.Stream()
    outs = []
    for t in (a, a.flip(0).contiguous()):
        with torch.cuda.stream(s):
            s.wait_stream(torch.cuda.default_stream())
            outs.append(neighbor_list(t, 4.0, None, True))
        s.synchronize()
    want = [neighbor_list(t, 4.0, None, True) for t in (a, a.flip(0).contiguous())]
    for got, ref in zip(outs, want):
        assert all(torch.equal(x, y) for x, y in zip(got, ref))


@pytest.mark.parametrize("dtype,cut", [(np.float32, 1e20), (np.float64, 1e200)])
def test_cutoff_whose_square_overflows(dtype, cut):
    """Every pair of an open system that takes the cell scan (lanes past its candidates match nothing)."""
    pos = np.random.default_rng(5).uniform(0, 30, (2100, 3)).astype(dtype)
    empty = torch.empty((0, 0), dtype=torch.from_numpy(pos).dtype, device=DEV)
    for full in (False, True):
        i, j, _, _, r = (t.cpu().numpy() for t in ops.neighbor_list(torch.from_numpy(pos).to(DEV), cut, empty, full))
        wi, wj = np.nonzero(~np.eye(len(pos), dtype=bool) if full else np.tri(len(pos), k=-1, dtype=bool))
        assert np.array_equal(i, wi) and np.array_equal(j, wj)
        want = np.linalg.norm((pos[wi] - pos[wj]).astype(np.float64), axis=1)
        np.testing.assert_allclose(r, want, rtol=8 * np.finfo(dtype).eps)
