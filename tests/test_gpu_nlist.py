"""The neighbour count from copies in bin order (lists of 8000 atoms and more)
against the count by atom index and against brute force: every integer equal,
separations bit for bit between the two."""
import numpy as np
import pytest
import torch
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu
RC = 4.3


def _gas(n, rng):
    """Clusters of 1 to 150 atoms smaller than the cutoff, 20 apart: centres
    with 0 to 149 images (one to a lane, two to a lane, past the LDS list)."""
    size = rng.integers(1, 151, n)
    owner = np.repeat(np.arange(n), size)[:n]
    side = int(np.ceil((owner.max() + 1) ** (1 / 3)))
    at = np.stack([owner % side, owner // side % side, owner // side**2], 1) * 20.0
    order = rng.permutation(n)
    return [(at + rng.uniform(0, 2.4, (n, 3)))[order]], [np.eye(3) * (side * 20.0 + 50.0)], [np.zeros(3, bool)]


def _cells(n, rng):
    """Sheared cells of 1 to 60 atoms, the small ones less than a cutoff
    across and with one open direction now and then; atoms outside the cell."""
    pos, cells, pbcs = [], [], []
    while sum(len(p) for p in pos) < n:
        k = min(int(rng.integers(1, 61)), n - sum(len(p) for p in pos))
        cell = np.eye(3) * (k / 0.066) ** (1 / 3) @ (np.eye(3) + rng.uniform(-0.2, 0.2, (3, 3)))
        pos.append((rng.uniform(-0.7, 1.7, (k, 3))) @ cell)
        cells.append(cell)
        pbcs.append(np.ones(3, bool) if rng.random() < 0.8 else rng.random(3) < 0.5)
    return pos, cells, pbcs


def _brute(pos, cell):
    T = np.array(np.meshgrid(*[range(-4, 5)] * 3, indexing="ij")).reshape(3, -1).T
    d = pos[None, :, None] + (T @ cell)[None, None] - pos[:, None, None]
    d2 = (d * d).sum(-1)
    d2[np.arange(len(pos)), np.arange(len(pos)), (T == 0).all(1).argmax()] = np.inf
    i, j, t = np.nonzero(d2 < RC * RC)
    o = np.lexsort((T[t, 2], T[t, 1], T[t, 0], j, i))
    return i[o], j[o], T[t][o]


@pytest.mark.parametrize("kind,n", [("gas", 7999), ("gas", 8000), ("gas", 8063), ("cells", 8001), ("cells", 9000)])
def test_count_from_bin_order(kind, n):
    from pyxtal_ff_amd import _native as nat
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(n)
    pos, cells, pbcs = (_gas if kind == "gas" else _cells)(n, rng)
    nl = DeviceNeighborList(pos, cells, pbcs, RC)
    i, j, T, r = (t.cpu() for t in nl.images())
    # the two-phase build without slots, by atom index
    b, ws, p, L = nl.builder, nl.builder._ws, nat.ptr, nat.lib()
    count = torch.empty_like(nl._img_count)
    geo = (p(nl.pos), n, p(nl.atom_struct), p(nl.atom_start), p(nl.cells))
    nat.check(L.pxff_nlist_count(*geo, p(nl.inv_cells), p(nl.pbc), p(nl.geom), max(b.nbins, 1), RC, p(ws["bin_count"]),
                                 p(ws["bin_start"]), p(ws["atom_bin"]), p(ws["wrap"]), p(ws["bin_atoms"]), p(count),
                                 nat.stream()), "count")
    assert torch.equal(count, nl._img_count)
    k = nl.nimg
    a, c = torch.empty(k, dtype=torch.int64, device="cuda"), torch.empty(k, dtype=torch.int64, device="cuda")
    t, s = torch.empty(3 * k, dtype=torch.int32, device="cuda"), torch.empty(3 * k, dtype=torch.float64, device="cuda")
    rows = torch.empty_like(nl._row_count)
    nat.check(L.pxff_nlist_fill(*geo, p(nl.pbc), p(nl.geom), RC, p(ws["bin_start"]), p(ws["atom_bin"]), p(ws["wrap"]),
                                p(ws["bin_atoms"]), p(nl.img_start), p(a), p(c), p(t), p(s), p(rows), nat.stream()), "fill")
    assert torch.equal(a.cpu(), i) and torch.equal(c.cpu(), j)
    assert torch.equal(t.cpu().view(-1, 3), T) and torch.equal(s.cpu().view(-1, 3), r)
    assert torch.equal(rows, nl._row_count)
    if kind == "gas":
        assert len(i) == 2 * len(cKDTree(pos[0]).query_pairs(RC, output_type="ndarray"))
        return
    first = np.concatenate([[0], np.cumsum([len(q) for q in pos])])
    # cells of 8 atoms and more: every translation in reach is one of -4..4
    for q in [q for q in range(len(pos)) if len(pos[q]) >= 8 and pbcs[q].all()][:40]:
        lo, hi = int(nl.img_start[first[q]]), int(nl.img_start[first[q + 1]])
        bi, bj, bT = _brute(pos[q], cells[q])
        assert np.array_equal(i[lo:hi].numpy() - first[q], bi) and np.array_equal(j[lo:hi].numpy() - first[q], bj)
        assert np.array_equal(T[lo:hi].numpy(), bT)
