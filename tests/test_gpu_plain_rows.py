"""Kernels of the plain (materialised rows) path against plain PyTorch sums
of the same terms.  Tolerance: FP64 sums of at most a few hundred terms of
both signs in another order, 1e-13 of the norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


# ten components per pass, two passes per turn; four atoms per workgroup
@pytest.mark.parametrize("n,nb", [(1, 1), (3, 9), (4, 10), (5, 11), (7, 20), (129, 21), (64, 30), (33, 55), (2, 400)])
def test_voigt_contract(n, nb):
    from pyxtal_ff_amd import so4
    g = torch.Generator().manual_seed(n + 1000 * nb)
    beta = torch.randn((n, nb), dtype=torch.float64, generator=g)
    rv = torch.randn((n, nb, 6), dtype=torch.float64, generator=g)
    ref = -(beta.unsqueeze(2) * rv).sum(1)
    out = so4.voigt_contract(beta.cuda(), rv.cuda()).cpu()
    assert out.shape == (n, 6) and _rel(out, ref) < 1e-13
    # operands off the natural layout are copied first
    bt = beta.t().contiguous().cuda().t()
    assert torch.equal(so4.voigt_contract(bt, rv.cuda()).cpu(), out)


def _list(kind):
    import numpy as np
    from pyxtal_ff_amd import workloads
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(7)
    if kind == "one":  # no images
        pos, cell, pbc, rc = np.zeros((1, 3)), np.eye(3) * 20.0, [False] * 3, 4.0
    elif kind == "small":  # self images, several images to a row
        pos, cell, pbc, rc = rng.uniform(0, 3.0, (3, 3)), np.eye(3) * 3.0, [True] * 3, 5.0
    elif kind == "cluster":  # 99 rows of one image, another atom out of reach
        pos, cell, pbc, rc = rng.uniform(0, 2.6, (100, 3)), np.eye(3) * 50.0, [False] * 3, 4.9
        pos[57] = 25.0
    else:
        s = workloads.amorphous_sio2(30, 61, seed=3)
        pos, cell, pbc, rc = s.positions, s.cell, s.pbc, 4.6
    return DeviceNeighborList([pos], [cell], [np.asarray(pbc)], rc).resolve()


@pytest.mark.parametrize("kind", ["one", "small", "cluster", "sio"])
@pytest.mark.parametrize("nb", [1, 21, 22, 43, 55])  # 64 columns (b, c) to a wavefront
def test_rows(kind, nb):
    from pyxtal_ff_amd import so4
    nl = _list(kind)
    ne, nr, n = nl.nimg, nl.nrows, nl.natoms
    g = torch.Generator().manual_seed(nb)
    db = torch.randn((max(ne, 1), nb, 3), dtype=torch.float64, generator=g)
    seq, r = nl.seq_array().cpu(), nl.img_r[: 3 * ne].view(-1, 3).cpu()
    pos, iv = nl.pos.view(-1, 3).cpu(), nl.inv_vol.cpu()
    row = nl.row_img.cpu()
    e_row = torch.repeat_interleave(torch.arange(nr), row[1 : nr + 1] - row[:nr])
    i = seq[e_row, 0]
    rowsum = torch.zeros((nr, nb, 3), dtype=torch.float64).index_add_(0, e_row, db[:ne])
    own = seq[:, 0] == seq[:, 1]
    dx_ref = rowsum.clone()
    dx_ref[own] = 0
    dx_ref[own] = -torch.zeros((n, nb, 3), dtype=torch.float64).index_add_(0, seq[:, 0], dx_ref)
    # bstress[row] -= Rj (x) dB, bstress[nsite] += Ri (x) dB
    bs = torch.zeros((nr, nb, 3, 3), dtype=torch.float64)
    bs.index_add_(0, e_row, -(r + pos[i])[:, None, :, None] * db[:ne, :, None, :])
    ns = nl.nsite.cpu()
    bs.index_add_(0, ns[i], pos[i][:, None, :, None] * db[:ne, :, None, :])
    rd_ref = -bs * iv[seq[:, 0]][:, None, None, None]
    rv_ref = torch.zeros((n, nb, 3, 3), dtype=torch.float64).index_add_(
        0, i, r[:, None, :, None] * db[:ne, :, None, :]) * iv[:, None, None, None]
    rv_ref = rv_ref.view(n, nb, 9)[:, :, [0, 4, 8, 1, 2, 5]]
    dbd = db.cuda().contiguous()
    dx, rd = so4.rows(nl, nb, dbd, stress=True)
    dx1, none = so4.rows(nl, nb, dbd, stress=False)
    dx2, rv = so4.rows_voigt(nl, nb, dbd)
    assert none is None and torch.equal(dx, dx1) and torch.equal(dx, dx2)
    for a, ref in ((dx, dx_ref), (rd, rd_ref), (rv, rv_ref)):
        assert a.shape == ref.shape
        if ref.any():
            assert _rel(a.cpu(), ref) < 1e-13
        else:
            assert not a.cpu().any()
    assert _rel(so4.rdxdr_reduce(nl, nb, rd), rv) < 1e-10 if ne else True  # the positions cancel


# 64 images to a pass of the wavefront: centres below, at and past one and two
# passes; the own row first, last and in between, with images of its own and
# without; an isolated atom
@pytest.mark.parametrize("kind", ["one", "small", "tiny", "cluster", "sio", 64, 65, 66, 129, 130])
def test_row_index(kind):
    import numpy as np
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    if isinstance(kind, int):  # every atom sees the others
        pos = np.random.default_rng(kind).uniform(0, 2.6, (kind, 3))
        nl = DeviceNeighborList([pos], [np.eye(3) * 50.0], [np.zeros(3, bool)], 4.9).resolve()
    elif kind == "tiny":  # one atom, all images its own, several passes
        nl = DeviceNeighborList([np.zeros((1, 3))], [np.eye(3) * 1.5], [np.ones(3, bool)], 5.0).resolve()
    else:
        nl = _list(kind)
    start, j = nl.img_start.cpu().numpy(), nl.img_j.cpu().numpy()
    seq, row_img, img_row, nsite = [], [], [], []
    for i in range(nl.natoms):
        mine = j[start[i]: start[i + 1]]
        for k in np.unique(np.append(mine, i)):
            if k == i:
                nsite.append(len(seq))
            row_img.append(start[i] + np.searchsorted(mine, k))
            img_row += [len(seq)] * int((mine == k).sum())
            seq.append((i, k))
    row_img.append(nl.nimg)
    n = len(seq)
    assert nl.nrows == n and np.array_equal(nl.seq_array().cpu().numpy(), np.array(seq))
    assert np.array_equal(nl.row_img.cpu().numpy()[: n + 1], row_img)
    assert np.array_equal(nl.img_row.cpu().numpy()[: nl.nimg], np.array(img_row, dtype=np.int64))
    assert np.array_equal(nl.nsite.cpu().numpy(), nsite)


@pytest.mark.parametrize("stress", [False, True])
@pytest.mark.parametrize("structures", [0, 1, 2])
def test_plain_path_without_atoms(structures, stress):
    """Energy, forces and stress of lists of no atoms: zeros, no error."""
    import numpy as np
    from pyxtal_ff_amd import potential, so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    nl = DeviceNeighborList([np.zeros((0, 3))] * structures, np.tile(np.eye(3) * 9.0, (structures, 1, 1)),
                            np.ones((structures, 3), dtype=bool), 4.9)
    cfg = so4.So4Config(4, 4.9, 0.99363)
    w = torch.ones(0, dtype=torch.float64, device="cuda")
    model = potential.NNPotential(["Si"], cfg.nb).cuda()
    species = [("Si", torch.zeros(0, dtype=torch.int64, device="cuda"))]
    out = potential.energy_forces_plain(nl, cfg, w, w, model, species, stress=stress)
    assert float(out["energy"]) == 0.0 and out["forces"].shape == (0, 3) and out["atom_energies"].shape == (0,)
    if stress:
        assert torch.equal(out["stress_voigt"].cpu(), torch.zeros(6, dtype=torch.float64))
