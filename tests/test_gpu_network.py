"""The fused network kernel (pxff_mlp_energy_grad: per-element networks
forward and backward to dE/dx) against torch autograd on the same
parameters: three elements mixed over 300 atoms, narrow and deep / wide
networks (up to 8 layers of 64), a 147-long descriptor (SO3 nmax = lmax =
6: the matrix-core kernel with more than 64 KB of LDS), and atoms without a
network."""
import numpy as np
import pytest
import torch

from pyxtal_ff_amd import potential
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _torch_reference(model, x, symbols):
    xr = x.detach().clone().requires_grad_(True)
    sp = potential.species_index(symbols, model.elements, x.device)
    e = model.atom_energies(xr, sp)
    (g,) = torch.autograd.grad(e.sum(), [xr])
    return e.detach(), g


@pytest.mark.parametrize("hidden,act,nin", [((30, 30), "Tanh", 55), ((24, 16, 8), "Softplus", 55),
                                            ((64,) * 7, "ELU", 55), ((30, 30), "Tanh", 147)])
def test_fused_network_matches_autograd(hidden, act, nin):
    rng = np.random.default_rng(5)
    n = 300
    symbols = list(rng.choice(["O", "Si", "C"], size=n, p=[0.5, 0.4, 0.1]))
    x = torch.as_tensor(rng.random((n, nin)), dtype=torch.float64, device="cuda")
    dr = {e: np.stack([np.full(nin, -0.1), np.full(nin, 1.2)], 1) for e in ("O", "Si", "C")}
    model = potential.NNPotential(["O", "Si", "C"], nin, hidden, seed=7, drange=dr, activation=act).cuda()
    with torch.no_grad():
        for p in model.parameters():
            p.add_(0.05 * torch.randn_like(p))
    sp_atom = potential.species_atom(symbols, model.elements, "cuda")
    e, beta = model.energy_grad(x, sp_atom)
    e_ref, g_ref = _torch_reference(model, x, symbols)
    print("hidden", hidden, act, "rel err e", rel_err(e.cpu().numpy(), e_ref.cpu().numpy()),
          "beta", rel_err(beta.cpu().numpy(), g_ref.cpu().numpy()), flush=True)
    assert rel_err(e.cpu().numpy(), e_ref.cpu().numpy()) < 1e-13
    assert rel_err(beta.cpu().numpy(), g_ref.cpu().numpy()) < 1e-12


def test_fused_network_unknown_species_gives_nan():
    n, nin = 70, 10
    x = torch.rand((n, nin), dtype=torch.float64, device="cuda")
    model = potential.NNPotential(["Si"], nin, (8,), seed=1).cuda()
    sp = torch.zeros(n, dtype=torch.int64, device="cuda")
    sp[3] = 5
    e, beta = model.energy_grad(x, sp)
    assert torch.isnan(e[3]) and torch.isnan(beta[3]).all()
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[3] = False
    assert torch.isfinite(e[keep]).all() and torch.isfinite(beta[keep]).all()


@pytest.mark.parametrize("elements,hidden,act", [(["Si"], (30, 30), "Tanh"), (["O", "Si", "C"], (24, 16, 8), "ReLU"),
                                                 (["O", "Si"], (), "Tanh"), (["O", "Si"], (64,) * 7, "Sigmoid")])
def test_energy_and_gradient_matches_autograd(elements, hidden, act):
    """The parameters taken at the call, compact rows per element: atoms
    without a network stay zero, parameters changed through .data or replaced
    are seen, and a model the kernel cannot stand for goes through autograd
    (a hooked layer, a subclass).  Tolerances as for the packed kernel."""
    nin, n = 21, 77
    rng = np.random.default_rng(len(elements))
    symbols = list(rng.choice(elements + ["H"], size=n))
    dr = {e: np.stack([np.full(nin, -0.1), np.full(nin, 1.2)], 1) for e in elements}
    model = potential.NNPotential(elements, nin, hidden, seed=7, drange=dr, activation=act).cuda()
    x = torch.as_tensor(rng.random((n, nin)), dtype=torch.float64, device="cuda")
    species = potential.species_index(symbols, model.elements, "cuda")

    def same(m):
        e, g = potential.energy_and_gradient(m, x, species)
        e_ref, g_ref = _torch_reference(m, x, symbols)
        assert not e.requires_grad and not g.requires_grad
        assert rel_err(e.cpu().numpy(), e_ref.cpu().numpy()) < 1e-13
        assert rel_err(g.cpu().numpy(), g_ref.cpu().numpy()) < 1e-12
        return e

    assert potential._networks(model, x, species) is not None
    e0 = same(model)
    lin = model.models[elements[0]].layers[0]
    lin.weight.data.mul_(1.5)  # bumps no version
    e1 = same(model)
    assert not torch.equal(e0, e1)
    lin.weight = torch.nn.Parameter(0.5 * lin.weight.detach())
    assert not torch.equal(e1, same(model))
    h = lin.register_forward_hook(lambda mod, a, out: 2.0 * out)
    assert potential._networks(model, x, species) is None
    same(model)
    h.remove()
    covered = [s for s in symbols if s in elements]
    keep = torch.as_tensor([k for k, s in enumerate(symbols) if s in elements], device="cuda")
    xs = x[keep].contiguous()
    sp = potential.species_index(covered, model.elements, "cuda")
    at = potential.species_atom(covered, [e for e, _ in sp], "cuda")
    a, b = potential.energy_and_gradient(model, xs, sp, at), potential.energy_and_gradient(model, xs, sp)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    with torch.no_grad():  # refused, as autograd refuses it
        with pytest.raises(RuntimeError):
            potential.energy_and_gradient(model, x, species)

    class Other(potential.NNPotential):
        pass

    model.__class__ = Other
    assert potential._networks(model, x, species) is None


# neurons around the 16-wide tiles and the splits of their sums (1 to 4 tiles),
# inputs around the 64-column groups and past the three held in registers, the
# deep and long ones with fewer partial tiles than wavefronts or another
# kernel; atoms below, at and past a tile, and without a network
@pytest.mark.parametrize("hidden,nin", [((), 1), ((1,), 3), ((16, 17), 64), ((32, 33), 65), ((48, 49), 192),
                                        ((64, 5), 193), ((20,), 400), ((30, 30, 30, 30), 260), ((24, 24), 250)])
@pytest.mark.parametrize("n", [1, 16, 33])
def test_network_tile_edges(hidden, nin, n):
    """Tolerances as above."""
    rng = np.random.default_rng(nin)
    model = potential.NNPotential(["Si", "O"], nin, hidden, seed=3).cuda()
    with torch.no_grad():
        for p in model.parameters():
            p.add_(0.05 * torch.randn_like(p))
    x = torch.as_tensor(rng.random((n, nin)), dtype=torch.float64, device="cuda")
    sp = torch.as_tensor(rng.integers(0, 2, n), device="cuda")
    symbols = [model.elements[int(k)] for k in sp.cpu()]
    if n == 33:
        sp[7] = -1
        symbols[7] = "H"
    e, beta = model.energy_grad(x, sp)
    e_ref, g_ref = _torch_reference(model, x, symbols)
    if n == 33:
        assert torch.isnan(e[7]) and torch.isnan(beta[7]).all()
        e[7], beta[7] = 0.0, 0.0
    assert rel_err(e.cpu().numpy(), e_ref.cpu().numpy()) < 1e-13
    assert rel_err(beta.cpu().numpy(), g_ref.cpu().numpy()) < 1e-12


# more 16-atom tiles than the chip holds at once in eight-wavefront workgroups
# (512 on 256 CUs): tiles of four wavefronts for short inputs and narrow layers
@pytest.mark.parametrize("n,nin,hidden,act", [(8193, 30, (30, 30), "Tanh"), (12001, 14, (16,), "Softplus"),
                                              (12288, 31, (17, 5), "ELU"), (24007, 5, (), "Tanh"),
                                              (8209, 91, (30, 30), "Sigmoid"), (16384, 91, (30, 30), "Tanh")])
def test_fused_network_many_tiles(n, nin, hidden, act):
    """Elements mixed within the tiles and sorted, an atom without a network,
    a last tile of one atom; tolerances as for few tiles."""
    rng = np.random.default_rng(n)
    model = potential.NNPotential(["O", "Si", "C"], nin, hidden, seed=7, activation=act).cuda()
    x = torch.as_tensor(rng.random((n, nin)), dtype=torch.float64, device="cuda")
    symbols = rng.choice(["O", "Si", "C"], size=n, p=[0.5, 0.4, 0.1])
    for order in (np.arange(n), np.argsort(symbols, kind="stable")):
        sy = list(symbols[order])
        e_ref, g_ref = _torch_reference(model, x, sy)
        sp = potential.species_atom(sy, model.elements, "cuda")
        sp[n // 2] = -1
        e, beta = model.energy_grad(x, sp)
        assert torch.isnan(e[n // 2]) and torch.isnan(beta[n // 2]).all()
        e[n // 2], beta[n // 2] = e_ref[n // 2], g_ref[n // 2]
        assert rel_err(e.cpu().numpy(), e_ref.cpu().numpy()) < 1e-13
        assert rel_err(beta.cpu().numpy(), g_ref.cpu().numpy()) < 1e-12
