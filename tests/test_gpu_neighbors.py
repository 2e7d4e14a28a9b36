"""Neighbour lists against a host search with the reference's rounded predicate
(neighbor_full.cpp:10-76, neighbor_half.cpp:10-100): the same pairs, order and
difference vectors, bit for bit, at the sizes where a wave, a workgroup, the
translation bits, the cell list or its sort keys change form."""

import numpy as np
import pytest

from pypolymlp_amd import capi

pytestmark = pytest.mark.gpu


def host_lists(axis, pos, rc, half):
    tr, prev = capi.cell_translations(axis, pos, rc)
    n = pos.shape[1]
    off, nb, tid, dd = [0], [], [], []
    for i in range(n):
        js = np.arange(i if half else n)
        d = (prev[:, js] - prev[:, i:i + 1]).T[:, None, :] + tr[None]
        r2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
        j, t = np.nonzero((r2 < rc * rc) & (r2 > 1e-20))
        nb.append(js[j]), tid.append(t), dd.append(d[j, t])
        if half:
            r2 = (tr[:, 0] * tr[:, 0] + tr[:, 1] * tr[:, 1]) + tr[:, 2] * tr[:, 2]
            x, y, z = tr.T
            tol = 1e-10
            up = (z >= tol) | ((np.abs(z) < tol) & (y >= tol)) | \
                ((np.abs(z) < tol) & (np.abs(y) < tol) & (x >= tol))
            t = np.nonzero((r2 < rc * rc) & (r2 > 1e-20) & up)[0]
            nb.append(np.full(len(t), i)), tid.append(t), dd.append(tr[t])
        off.append(sum(len(v) for v in nb[-2 if half else -1:]) + off[-1])
    return np.array(off), np.concatenate(nb), np.concatenate(tid), np.concatenate(dd)


def cell(n, box, seed, skew=0.0):
    rng = np.random.default_rng(seed)
    axis = np.diag(np.array(box, dtype=float))
    axis[0, 1] = skew * box[1]
    return axis, axis @ rng.uniform(-0.2, 1.2, size=(3, n))


CASES = {
    # (atoms, box, cutoff, skew): 1 atom with many translations; around one wave,
    # one workgroup and its second round; more and fewer than 128 translations
    "one": (1, (2.5, 2.7, 2.9), 6.0, 0.0),
    "two_skew": (2, (3.0, 3.1, 3.3), 7.0, 0.3),
    "wave-1": (63, (9.0, 9.0, 9.0), 5.0, 0.0),
    "wave": (64, (9.0, 9.5, 9.0), 5.0, 0.2),
    "wave+1": (65, (9.0, 9.0, 30.0), 5.0, 0.0),
    "flat_129": (129, (4.0, 25.0, 9.0), 6.0, 0.0),
    "group-1": (255, (16.0, 14.0, 13.0), 6.0, 0.0),
    "group+1": (257, (16.0, 14.0, 13.0), 6.0, 0.1),
    # from 1,024 atoms on by bins where three fit each direction, else all pairs
    "bins_3": (1024, (18.5, 18.2, 18.3), 6.0, 0.0),
    "bins_skew": (1100, (20.0, 25.0, 19.0), 6.0, 0.15),
    "thin": (1030, (40.0, 40.0, 9.0), 6.0, 0.0),
}


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("name", sorted(CASES))
def test_lists_bit_exact(name, half):
    n, box, rc, skew = CASES[name]
    axis, pos = cell(n, box, 3, skew)
    got = capi.neighbor(axis, pos, rc, half=half)
    want = host_lists(axis, pos, rc, half)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


@pytest.mark.parametrize("n", [2048, 2050])
def test_dense_cluster_sort_keys(n):
    """An atom with as many neighbours as LDS holds sort keys, and with more."""
    rng = np.random.default_rng(n)
    axis = np.diag([13.0, 13.0, 13.0])
    pos = 5.0 + rng.uniform(0.0, 1.0, size=(3, n))
    off, nb, tid, d = capi.neighbor(axis, pos, 4.0)
    assert np.array_equal(np.diff(off), np.full(n, n - 1))
    full = np.arange(n)
    for i in (0, 1, n // 2, n - 1):
        seg = slice(off[i], off[i + 1])
        assert np.array_equal(nb[seg], full[full != i])
        assert np.array_equal(d[seg], (pos[:, nb[seg]] - pos[:, i:i + 1]).T)
    hoff, hnb, _, hd = capi.neighbor(axis, pos, 4.0, half=True)
    assert np.array_equal(np.diff(hoff), full)
    keep = nb < np.repeat(full, n - 1)
    assert np.array_equal(hnb, nb[keep]) and np.array_equal(hd, d[keep])


@pytest.mark.parametrize("name", ["bins", "thin"])
def test_lists_beyond_one_scan_round(name):
    """More atoms than one round of the offsets' prefix sum (4,096), by both
    searches: some atoms' lists against the host, and every pair from both ends."""
    n, rc = 4500, 4.0
    axis, pos = cell(n, (34.0, 33.0, 32.0) if name == "bins" else (95.0, 95.0, 4.0), 5)
    off, nb, tid, d = capi.neighbor(axis, pos, rc)
    assert off[-1] == len(nb) and np.all(np.diff(off) >= 0)
    tr, p = capi.cell_translations(axis, pos, rc)
    for i in (0, 1, 1023, 4094, 4095, 4096, 4097, n - 1):
        v = (p - p[:, i:i + 1]).T[:, None, :] + tr[None]
        r2 = (v[..., 0] * v[..., 0] + v[..., 1] * v[..., 1]) + v[..., 2] * v[..., 2]
        j, t = np.nonzero((r2 < rc * rc) & (r2 > 1e-20))
        seg = slice(off[i], off[i + 1])
        assert np.array_equal(nb[seg], j) and np.array_equal(tid[seg], t)
        assert np.array_equal(d[seg], v[j, t])
    i = np.repeat(np.arange(n), np.diff(off))
    assert np.array_equal(np.sort(i * n + nb), np.sort(nb * n + i))
    hoff, hnb, _, hd = capi.neighbor(axis, pos, rc, half=True)
    low = nb < i
    own = hnb == np.repeat(np.arange(n), np.diff(hoff))
    assert np.array_equal(hnb[~own], nb[low]) and np.array_equal(hd[~own], d[low])
