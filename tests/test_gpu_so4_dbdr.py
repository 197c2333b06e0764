"""The matrix-core dB/dr kernel against the per-image kernel at the edges of
its tiles and passes: 16 images to a tile, 48 (2J = 10: 32) to the first
pass, the rest in passes of the persistent kernel.

Tolerance: both sum the same FP64 terms in another order, a few hundred per
output, with rows of at most unit size: 1e-13 of the whole (norm), 1e-12 of
the largest element for any single one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# every centre of a cluster smaller than the cutoff has n - 1 images; 1 atom
# (none) and 2 (one image) are the smallest
@pytest.mark.parametrize("twol", [0, 2, 6, 8, 10])
@pytest.mark.parametrize("n", [1, 2, 16, 17, 18, 33, 34, 49, 50, 98])
def test_dbdr_image_counts(n, twol):
    from pyxtal_ff_amd import so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(100 * twol + n)
    pos = rng.uniform(0.0, 2.6, (n, 3))
    nl = DeviceNeighborList([pos], [np.eye(3) * 100.0], [np.zeros(3, bool)], 4.9)
    assert nl.nimg == n * (n - 1)
    cfg = so4.So4Config(twol, 4.9, 0.99363)
    w = torch.rand(n, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda() + 0.5
    _, z, _ = so4.forward(nl, cfg, w, w)
    k = nl.nimg * cfg.nb * 3
    ref = so4.dbdr_per_image(nl, cfg, w, z)[:k]
    for atom_major in (False, True):
        d = so4.dbdr(nl, cfg, w, z, atom_major=atom_major)[:k]
        if k:
            assert float((d - ref).norm() / ref.norm()) < 1e-13
            assert float((d - ref).abs().max() / ref.abs().max()) < 1e-12


# 4096 atoms and more take the kernel with several centres per wavefront: 4, 5
# (rounded to 6 at 2J = 8), 12 and all of a wavefront's lane groups to a centre
@pytest.mark.parametrize("n,twol", [(4096, 8), (4097, 6), (5200, 8), (6500, 2), (12300, 8), (16500, 6), (8200, 4),
                                    (66000, 0)])
def test_utot_centres_per_wavefront(n, twol):
    """U_tot of the staged records against the kernel that stages in LDS, a
    wavefront per centre: a gas of clusters with 0 to 70 images per centre.
    Sums of at most 70 terms in another order, 1e-14 of the norm."""
    from pyxtal_ff_amd import so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(n)
    size = rng.integers(1, 72, n)  # atoms per cluster, clusters 20 apart
    owner = np.repeat(np.arange(n), size)[:n]
    side = int(np.ceil((owner.max() + 1) ** (1 / 3)))
    at = np.stack([owner % side, owner // side % side, owner // side**2], 1) * 20.0
    pos = at + rng.uniform(0, 2.4, (n, 3))
    nl = DeviceNeighborList([pos], [np.eye(3) * (side * 20.0 + 50.0)], [np.zeros(3, bool)], 4.3)
    assert nl.nimg > n
    cfg = so4.So4Config(twol, 4.3, 0.99363)
    w = torch.rand(n, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda() + 0.5
    a, b = so4.ui(nl, cfg, w, w), so4.ui(nl, cfg, w, w, staged=False)
    assert float((a - b).norm() / b.norm()) < 1e-14
    assert float((a - b).abs().max() / b.abs().max()) < 1e-13
    assert torch.equal(a, so4.ui(nl, cfg, w, w, torch.arange(n - 1, -1, -1, device="cuda")))
    # the tangent's sums, against its wavefront per centre (within its static workspace)
    if n * cfg.nhalf * 16 < 30e6:
        _, z, _ = so4.forward(nl, cfg, w, w)
        dr = torch.randn(nl.nimg * 3, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda()
        t = so4.tangent(nl, cfg, w, z, dr)
        ref = torch.empty_like(t)
        so4.tangent_noalloc(nl, cfg, w, z, dr, ref)
        assert float((t - ref).norm() / ref.norm()) < 1e-13


# one atom, the edges of a 64-atom tile, more tiles than XCDs, a last tile of one atom
@pytest.mark.parametrize("n,twol", [(1, 8), (2, 0), (63, 2), (64, 8), (65, 10), (513, 4), (577, 6)])
def test_tangent_b_against_dbdr(n, twol):
    """dB along displacements against the sum over images of dB/dr (sums of
    at most a few thousand FP64 terms: 1e-12 of the norm)."""
    from pyxtal_ff_amd import so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(n + twol)
    side = int(np.ceil(n ** (1 / 3)))
    at = np.stack(np.unravel_index(np.arange(n), (side,) * 3), 1) * 2.3
    pos = at + rng.uniform(0, 0.4, (n, 3))
    nl = DeviceNeighborList([pos], [np.eye(3) * (side * 2.3 + 50.0)], [np.zeros(3, bool)], 4.3)
    cfg = so4.So4Config(twol, 4.3, 0.99363)
    g = torch.Generator().manual_seed(n)
    w = torch.rand(n, dtype=torch.float64, generator=g).cuda() + 0.5
    dr = torch.randn(nl.nimg, 3, dtype=torch.float64, generator=g).cuda()
    _, z, _ = so4.forward(nl, cfg, w, w)
    db = so4.tangent(nl, cfg, w, z, dr).view(-1)[: n * cfg.nb].view(n, cfg.nb)
    per_image = so4.dbdr(nl, cfg, w, z)[: nl.nimg * cfg.nb * 3].view(nl.nimg, cfg.nb, 3)
    ref = torch.zeros_like(db).index_add(0, nl.img_atom[: nl.nimg], (per_image * dr[:, None, :]).sum(2))
    assert float((db - ref).norm()) <= 1e-12 * max(float(ref.norm()), 1e-300)


# the last list summed per component, the first per tile (its last tile one atom), and past it
@pytest.mark.parametrize("n,twol", [(12224, 4), (12225, 0), (12225, 10), (12288, 2), (12351, 8)])
def test_b_row_sums(n, twol):
    """B summed from the Z kernel's row partials against B from U_tot and Z
    (a few dozen FP64 terms in another order: 1e-13 of the norm)."""
    from pyxtal_ff_amd import so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(n + twol)
    side = int(np.ceil(n ** (1 / 3)))
    pos = np.stack(np.unravel_index(np.arange(n), (side,) * 3), 1) * 2.6 + rng.uniform(0, 0.4, (n, 3))
    nl = DeviceNeighborList([pos], [np.eye(3) * (side * 2.6 + 50.0)], [np.zeros(3, bool)], 3.5)
    cfg = so4.So4Config(twol, 3.5, 0.99363)
    w = torch.rand(n, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda() + 0.5
    b, z, u = so4.forward(nl, cfg, w, w)
    ref = so4.bi(nl, cfg, u, z)
    assert float((b - ref).norm() / ref.norm()) < 1e-13
    assert float((b[-1] - ref[-1]).norm() / ref[-1].norm()) < 1e-13


# five, four and one lane groups to a centre; a cap of no, one, some and all images
@pytest.mark.parametrize("n", [4096, 6001, 13000])
@pytest.mark.parametrize("part", [0.0, 1e-9, 0.37, 1.0])
def test_staged_tangent_stays_within_its_records(n, part):
    """pxff_so4_tangent_staged with room for `cap` records writes and reads
    none past them: the images after that add nothing, as with zero
    displacements (the sums only lose zeros: the same bits)."""
    from pyxtal_ff_amd import _native as nat, so4
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    rng = np.random.default_rng(n)
    side = int(np.ceil((n / 4) ** (1 / 3)))
    owner = np.arange(n) // 4
    at = np.stack([owner % side, owner // side % side, owner // side**2], 1) * 20.0
    pos = at + rng.uniform(0, 2.4, (n, 3))
    nl = DeviceNeighborList([pos], [np.eye(3) * (side * 20.0 + 50.0)], [np.zeros(3, bool)], 4.3)
    ne = nl.nimg
    cfg = so4.So4Config(4, 4.3, 0.99363)
    w = torch.rand(n, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda() + 0.5
    _, z, _ = so4.forward(nl, cfg, w, w)
    dr = torch.randn(ne * 3, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda()
    cap = int(np.ceil(part * ne))
    stage = torch.full((ne * 10,), float("nan"), dtype=torch.float64, device="cuda")
    du = torch.empty(2 * cfg.nhalf * 64 * ((n + 63) // 64), dtype=torch.float64, device="cuda")
    db = torch.empty((n, cfg.nb), dtype=torch.float64, device="cuda")
    p = nat.ptr
    nat.check(nat.lib().pxff_so4_tangent_staged(cfg.params, n, p(nl.img_start), p(nl.img_j), p(nl.img_r), p(w), p(dr),
                                                p(z), cap, p(stage), p(du), p(db), nat.stream()), "tangent")
    assert bool(stage[cap * 10:].isnan().all())
    dr[3 * cap:] = 0.0
    assert torch.equal(db, so4.tangent(nl, cfg, w, z, dr))
