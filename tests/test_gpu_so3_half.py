"""The m >= 0 kernels of the SO(3) energy + force path against the general
ones: the (image, l) accumulation, the per-output power spectrum, the full A
and the per-image adjoint with recomputed radial integrals.

Tolerances: the stored radial integrals (table or quadrature) and the
recomputed ones agree to about 1e-14 of each function's largest value, and a
sum over the (n, l, m) of an image loses at most about two digits more:
1e-12 for the expansion and P, 1e-11 for dE/dr (as the existing comparison of
stored with recomputed integrals)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a - b).norm() / b.norm())


# lmax = 0 (one lane), odd and even top l, the largest lmax, nmax past the table
@pytest.mark.parametrize("n,nmax,lmax", [(24, 1, 0), (33, 2, 1), (40, 4, 2), (31, 11, 3), (57, 3, 4), (53, 8, 5),
                                         (96, 6, 6)])
def test_so3_half_layout_equals_general_kernels(n, nmax, lmax):
    from pyxtal_ff_amd import _native as nat
    from pyxtal_ff_amd import so3 as d3
    from pyxtal_ff_amd import workloads
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    s = workloads.amorphous_sio2(n // 3, n - n // 3, seed=n)
    nl = DeviceNeighborList([s.positions], [s.cell], [s.pbc], 4.6).resolve()
    cfg = d3.So3Config(nmax, lmax, 4.6, 2.0)
    z = torch.as_tensor(s.numbers, device="cuda")
    p = nat.ptr
    ct = torch.empty(n * cfg.csz * 2, dtype=torch.float64, device="cuda")
    nat.check(nat.lib().pxff_so3_ctot(cfg.params, n, p(nl.img_start), p(nl.img_j), p(nl.img_r), p(z), p(cfg.G),
                                      p(cfg.rq), p(cfg.lnorm), None, p(ct), None, nat.stream()), "pxff_so3_ctot")
    beta = torch.randn((n, cfg.ncoef), dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda()
    a = d3.adjoint_a(nl, cfg, ct, beta)
    ref = d3.deidrj(nl, cfg, z, a)
    x, cth, rad = d3.forward_half(nl, cfg, z)
    full = ct.view(n, nmax, lmax + 1, 2 * lmax + 1, 2)
    half = torch.stack([full[:, :, l, lmax + m] for l in range(lmax + 1) for m in range(l + 1)], 2)
    assert _rel(cth.view(n, nmax, -1, 2), half) < 1e-12
    assert _rel(d3.ctot(nl, cfg, z), ct) < 1e-12
    assert _rel(x, d3.power(nl, cfg, ct)) < 1e-12
    d = d3.adjoint_half(nl, cfg, z, cth, beta, rad)()
    assert _rel(d, ref) < 1e-11
    dc = d3.adjoint_half(nl, cfg, z, cth, beta, rad, counted=True)()
    assert torch.equal(dc[: nl.nimg], d)
    assert _rel(d3.deidrj(nl, cfg, z, a, radial=rad), ref) < 1e-11
    # rows off a 16-byte boundary take the per-image kernel
    off = torch.empty(rad.numel() + 1, dtype=torch.float64, device="cuda")[1:]
    off.copy_(rad)
    assert _rel(d3.deidrj(nl, cfg, z, a, radial=off), ref) < 1e-11


@pytest.mark.parametrize("nmax,lmax", [(3, 4), (6, 6), (1, 0)])
def test_so3_direct_radial_store_equals_sorted(nmax, lmax):
    """The two evaluations of the radial table store the same bits."""
    from pyxtal_ff_amd import so3 as d3
    from pyxtal_ff_amd import workloads
    from pyxtal_ff_amd.neighbors import NeighborListBuilder
    s = workloads.amorphous_sio2(30, 61, seed=3)
    cfg = d3.So3Config(nmax, lmax, 5.0, 2.0)
    z = torch.as_tensor(s.numbers, device="cuda")
    pos = torch.as_tensor(s.positions, device="cuda")
    rows = []
    for cap in (65536, 65537):  # the largest capacity of the direct form, and past it
        b = NeighborListBuilder([len(s)], [s.cell], [s.pbc], 5.0)
        b.img_capacity = cap
        nl = b.build(pos).resolve()
        _, rad = d3.ctot(nl, cfg, z, radial=True)
        rows.append(rad[: nl.nimg * (lmax + 1) * 2 * nmax].clone())
    assert torch.equal(rows[0], rows[1])


@pytest.mark.parametrize("nmax,lmax", [(1, 0), (2, 1), (3, 4), (8, 5), (6, 6)])
def test_so3_adjoint_of_any_a(nmax, lmax):
    """dE/dr from a full A without the symmetry of the expansion: the same
    with the stored radial integrals as with recomputed ones, at every
    alignment of the store."""
    from pyxtal_ff_amd import so3 as d3
    from pyxtal_ff_amd import workloads
    from pyxtal_ff_amd.neighbors import DeviceNeighborList
    s = workloads.amorphous_sio2(11, 22, seed=nmax)
    nl = DeviceNeighborList([s.positions], [s.cell], [s.pbc], 4.6).resolve()
    n = nl.natoms
    cfg = d3.So3Config(nmax, lmax, 4.6, 2.0)
    z = torch.as_tensor(s.numbers, device="cuda")
    _, rad = d3.ctot(nl, cfg, z, radial=True)
    a = torch.randn(n * cfg.csz * 2, dtype=torch.float64, generator=torch.Generator().manual_seed(lmax)).cuda()
    ref = d3.deidrj(nl, cfg, z, a)
    off = torch.empty(rad.numel() + 1, dtype=torch.float64, device="cuda")[1:]
    off.copy_(rad)
    assert _rel(d3.deidrj(nl, cfg, z, a, radial=off), ref) < 1e-11
    assert _rel(d3.deidrj(nl, cfg, z, a, radial=rad), ref) < 1e-11
    counted = d3.deidrj(nl, cfg, z, a, radial=rad, counted=True)
    assert _rel(counted[: nl.nimg], ref) < 1e-11
