"""The binned 3-D deposits and fused Esirkepov phase (particles in any slot order) against the FP64 oracle: random
and cell order, both shapes, inactive slots, several species, fewer slots than a chunk and more, tiles that do not
divide the grid, steps of a cell or more, and particles outside the domain (their nodes leave the tile's box)."""

import numpy as np
import pytest
import torch

from oracle import pic_oracle as O
from pypic3d_amd import _native as N
from pypic3d_amd import _tensors as T
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc, make_species, particle_planes, pic_particles, tiled_particles_from_arrays
from pypic3d_amd.particles.particle_class import SpeciesConfig
from tests.gpu_helpers import TOL, gpu_field, host, host_particles, oracle_params, rel_err
from tests.helpers import random_field, random_particles, species

pytestmark = pytest.mark.gpu


def _setup(shape, sf, P, seed, vmax=0.3, spacing=0.5, pbc=(0, 0, 0), pusher="boris"):
    static, dyn = workloads.make_parameters(shape, d=(spacing,) * 3, dt=0.05, shape_factor=sf, pbc=pbc,
                                            particle_pusher=pusher)
    p = oracle_params(static, dyn)
    x, u, act = random_particles(p, S=2, P=P, seed=seed, vmax=vmax, inactive_frac=0.1)
    sp = species(2, charge=(-1.0, 2.0), mass=(1.0, 50.0), weight=(0.5, 0.25))
    cfg = SpeciesConfig(sp.charge, sp.mass, sp.weight, sp.update_x, sp.update_u)
    desc = make_desc(static, dyn)
    csp = make_species(cfg, P)
    return p, sp, desc, csp, x, u, act


def _workspace(desc, csp, kind):
    n = int(N.lib().pic_binned_workspace_bytes(desc, csp, kind))
    assert n > 0
    return torch.empty(n, dtype=torch.uint8, device="cuda")


def _deposit(kind, desc, csp, pp, p):
    J = [torch.zeros(p.shape, dtype=torch.float32, device="cuda") for _ in range(3)]
    ws = _workspace(desc, csp, kind)
    name = ("pic_deposit_rho_binned", "pic_deposit_direct_binned", "pic_deposit_esirkepov_binned")[kind]
    N.call(name, desc, csp, pp, N.ptr(J[0]) if kind == 0 else N.p3(J), N.ptr(ws), ws.numel(), N.stream_handle())
    return [host(c) for c in (J[:1] if kind == 0 else J)]


def _oracle(kind, x, u, act, sp, p):
    if kind == 0:
        return [O.rho_raw(x, act, sp, p)]
    return O.j_from_rhov_raw(x, u, act, sp, p) if kind == 1 else O.esirkepov_raw(x, u, act, sp, p)


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("sf", [1, 2])
@pytest.mark.parametrize("shape,P", [((8, 8, 8), 700), ((17, 9, 24), 3000), ((3, 40, 5), 1025)])
def test_binned_deposits_match_oracle(kind, sf, shape, P):
    # positions FP32-rounded on a spacing that FP32 does not hold exactly
    p, sp, desc, csp, x, u, act = _setup(shape, sf, P, 3, spacing=0.3)
    parts = tiled_particles_from_arrays(x, u, act)
    got = _deposit(kind, desc, csp, pic_particles(*particle_planes(parts)), p)
    for a, b in zip(got, _oracle(kind, x, u, act, sp, p)):
        assert rel_err(a, b) <= TOL


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("sf", [1, 2])
def test_binned_deposits_of_sorted_and_long_moving_particles(kind, sf):
    """Equal cells in neighbouring lanes, positions on cell faces, particles past the domain and steps of up to two
    and a half cells."""
    p, sp, desc, csp, x, u, act = _setup((9, 10, 11), sf, 2000, 5, vmax=2.5)
    order = np.lexsort((np.floor(x[0, :, 2] * 2), np.floor(x[0, :, 1] * 2), np.floor(x[0, :, 0] * 2)))
    x, u = x[:, order], u[:, order]
    x[0, :50] = np.round(x[0, :50] * 2) / 2
    x[1, :20, 0] = p.wind[0] / 2 + 0.3
    parts = tiled_particles_from_arrays(x, u, act)
    got = _deposit(kind, desc, csp, pic_particles(*particle_planes(parts)), p)
    for a, b in zip(got, _oracle(kind, x, u, act, sp, p)):
        assert rel_err(a, b) <= TOL


@pytest.mark.parametrize("sf,pusher,pbc", [(1, "boris", (0, 0, 0)), (1, "higuera_cary", (1, 2, 0)), (2, "boris", (2, 0, 1))])
@pytest.mark.parametrize("ext", [False, True])
def test_binned_fused_phase_matches_oracle(sf, pusher, pbc, ext):
    p, sp, desc, csp, x, u, act = _setup((12, 10, 9), sf, 2500, 11, vmax=0.05, pbc=pbc, pusher=pusher)   # |v| < 0.9 c
    E, B = ([random_field(p, s + c, scale=0.2) for c in range(3)] for s in (20, 30))
    Ex, Bx = ([random_field(p, s + c, scale=0.1) for c in range(3)] for s in (40, 50))
    parts = tiled_particles_from_arrays(x, u, act)
    xp, up, ac = particle_planes(parts)
    xs, xv = T.new_soa(2, 2500, "cuda")
    us, uv = T.new_soa(2, 2500, "cuda")
    ao = torch.empty_like(ac)
    g = lambda F: [gpu_field(c)[0, 0, 0].contiguous() for c in F]   # noqa: E731
    Eg, Bg, Exg, Bxg = g(E), g(B), g(Ex), g(Bx)
    J = [torch.zeros(p.shape, dtype=torch.float32, device="cuda") for _ in range(3)]
    ws = _workspace(desc, csp, 2)
    N.call("pic_fused_push_esirkepov_binned", desc, csp, pic_particles(xp, up, ac), N.p3(Eg), N.p3(Bg),
           N.p3(Exg) if ext else None, N.p3(Bxg) if ext else None,
           pic_particles([xs[0], xs[1], xs[2]], [us[0], us[1], us[2]], ao), N.p3(J), N.ptr(ws), ws.numel(),
           N.stream_handle())
    Et, Bt = ([a + b for a, b in zip(F, X)] if ext else F for F, X in ((E, Ex), (B, Bx)))
    un = O.particle_push(x, u, act, sp, Et, Bt, p)
    for c, want in enumerate(O.esirkepov_raw(x, un, act, sp, p)):
        assert rel_err(host(J[c]), want) <= TOL
    xn = O.update_positions(x, un, act, sp, p.dt)
    xn, un, an, _ = O.refresh_particles(xn, un, act, p)
    xg, ug, ag = host_particles(parts._replace(x=xv, u=uv, active=ao.view(1, 1, 1, 2, 2500)))
    np.testing.assert_array_equal(ag, an)
    assert np.max(np.abs(xg - xn)) <= 1e-6 * max(p.wind)
    assert rel_err(ug, un) <= TOL


def test_large_chunks_agree_with_small_ones_and_the_slot_ordered_kernel():
    """More than 2^21 slots take the large chunks; rho of the same particles through the atomics kernel."""
    static, dyn = workloads.make_parameters((40, 33, 50), d=(0.3,) * 3, dt=0.05)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(33, weight=0.01)], seed=2)
    xp, up, act = particle_planes(parts)
    assert act.numel() > 1 << 21
    desc, sp = make_desc(static, dyn), make_species(cfg, act.shape[1])
    shape = tuple(desc.dims)
    for perm in (None, torch.randperm(act.numel(), device="cuda")):
        if perm is not None:
            xp = [c.reshape(-1)[perm].reshape(c.shape) for c in xp]
            up = [c.reshape(-1)[perm].reshape(c.shape) for c in up]
        pp = pic_particles(xp, up, act)
        for kind, plain in ((0, "pic_deposit_rho"), (1, "pic_deposit_direct"), (2, "pic_deposit_esirkepov")):
            J = [torch.zeros(shape, dtype=torch.float32, device="cuda") for _ in range(3)]
            N.call(plain, desc, sp, pp, N.ptr(J[0]) if kind == 0 else N.p3(J), N.stream_handle())
            got = _deposit(kind, desc, sp, pp, oracle_params(static, dyn))
            for a, b in zip(got, J):
                assert rel_err(a, host(b)) <= TOL


@pytest.mark.parametrize("shape", [(16, 1, 1), (16, 16, 1), (1, 8, 8)])
def test_grids_without_three_axes_have_no_bins(shape):
    static, dyn = workloads.make_parameters(shape, dt=0.05)
    sp = make_species(SpeciesConfig([1.0], [1.0], [1.0], [[True] * 3], [[True] * 3]), 10)
    assert N.lib().pic_binned_workspace_bytes(make_desc(static, dyn), sp, 2) == -1
    assert T.binned_workspace(make_desc(static, dyn), sp, 2, "cuda") is None


@pytest.mark.parametrize("order", ["random", "cell"])
@pytest.mark.parametrize("sf", [1, 2])
@pytest.mark.parametrize("ext", [False, True])
def test_push_and_fused_phase_through_tiles_equal_the_slot_ordered_kernels(order, sf, ext):
    """Enough slots for the push through tiles: random order takes it, cell order the push in slot order; both against
    pic_push (same stencils; the sums may be ordered differently, so a few ulp of |v| <= 1) and the plain deposit."""
    static, dyn = workloads.make_parameters((21, 16, 30), d=(0.3,) * 3, dt=0.05, shape_factor=sf, pbc=(0, 2, 1))
    p = oracle_params(static, dyn)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(30, weight=0.01, vth=(0.1,) * 3)], seed=2)
    xp, up, act = particle_planes(parts)
    n = act.numel()
    assert n > 1 << 18
    act = act.clone()
    act[0, ::17] = False
    if order == "random":
        perm = torch.randperm(n, device="cuda")
        xp, up = [[c.reshape(-1)[perm].reshape(c.shape).contiguous() for c in q] for q in (xp, up)]
    xp[1][0, 100] = 0.5 * p.wind[1] + 0.05       # outside: its nodes leave every tile's box
    desc, sp = make_desc(static, dyn), make_species(cfg, n)
    g = lambda s: [gpu_field(random_field(p, s + c, scale=0.2))[0, 0, 0].contiguous() for c in range(3)]   # noqa: E731
    E, B, Ex, Bx = g(1), g(4), g(7), g(10)
    Ee, Be = (N.p3(Ex), N.p3(Bx)) if ext else (None, None)
    pp, s = pic_particles(xp, up, act), N.stream_handle()
    want, got = (torch.empty((3, 1, n), dtype=torch.float32, device="cuda") for _ in range(2))
    N.call("pic_push", desc, sp, pp, N.p3(E), N.p3(B), Ee, Be, N.p3(want), s)
    ws = _workspace(desc, sp, T.PUSH)
    N.call("pic_push_binned", desc, sp, pp, N.p3(E), N.p3(B), Ee, Be, N.p3(got), N.ptr(ws), ws.numel(), s)
    assert float((got - want).abs().max()) <= 8 * 2.0 ** -23
    J = [torch.zeros(p.shape, dtype=torch.float32, device="cuda") for _ in range(6)]
    N.call("pic_deposit_esirkepov", desc, sp, pic_particles(xp, [want[a] for a in range(3)], act), N.p3(J[:3]), s)
    xo, uo = (torch.empty((3, 1, n), dtype=torch.float32, device="cuda") for _ in range(2))
    ao = torch.empty_like(act)
    ws = _workspace(desc, sp, 2)
    N.call("pic_fused_push_esirkepov_binned", desc, sp, pp, N.p3(E), N.p3(B), Ee, Be, pic_particles(xo, uo, ao),
           N.p3(J[3:]), N.ptr(ws), ws.numel(), s)
    for a, b in zip(J[3:], J[:3]):
        assert rel_err(host(a), host(b)) <= TOL
    xw = torch.empty_like(xo)
    N.call("pic_advance_positions", desc, sp, pic_particles(xp, want, act), 1.0, N.p3(xw), s)
    aw = act.clone()
    N.call("pic_particle_boundaries", desc, sp, pic_particles(xw, want, aw), s)
    assert torch.equal(ao, aw)
    # an ulp of the velocity moves a position by dt ulp, at most one ulp of x after rounding; at a wall it mirrors
    assert float((xo - xw).abs().max()) <= 2.0 ** -21 and float((uo - want).abs().max()) <= 8 * 2.0 ** -23
