"""Tile-ordered fused kernel on grids whose lines are not FP32 numbers (FP64
anchors) against the strided tile kernel on the same launch: tiles that do not
divide the grid, every particle boundary, frozen axes, particles that drifted
out of their tile or lie on a face (rare list)."""

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import pic_particles
from pypic3d_amd.runner import ElectrodynamicRunner
from tests.gpu_helpers import gpu_field, oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu


def _launch(r, general):
    src, dst = r.cur, 1 - r.cur
    for c in r.J:
        c.zero_()
    r.tile_ws[0] = -7
    head = (r.desc, r.sp, r._pp(src), N.p3(r.E[r.ecur]), N.p3(r.B), r.Ee, r.Be, r._pp(dst), N.p3(r.J), r.tile,
            N.ptr(r.starts), r.rounds)
    if general:
        N.call("pic_fused_push_esirkepov_tiled_general", *head, N.ptr(r.tile_ws), N.stream_handle())
    else:
        N.call("pic_fused_push_esirkepov_tiled", *head, r.min_blocks, N.ptr(r.tile_ws), N.stream_handle())
    torch.cuda.synchronize()
    return (torch.stack(r.J).clone(), r.pos[dst].clone(), r.vel[dst].clone(), r.act[dst].clone(), int(r.tile_ws[0]))


@pytest.mark.parametrize("tile", [4, 8])
@pytest.mark.parametrize("n,wind,pbc,frozen", [
    ((13, 10, 9), (1.3, 0.7, 2.1), (0, 0, 0), False),
    ((8, 8, 8), (0.9, 0.3, 1.1), (0, 1, 2), False),
    ((5, 4, 17), (0.1, 0.6, 1.9), (2, 0, 1), True),
])
def test_general_grid_tile_kernel_agrees_with_strided_kernel(tile, n, wind, pbc, frozen):
    """Offsets from a node are FP64 differences in both kernels, rounded to
    FP32 after at most one further FP64 rounding: weights agree to 2^-24, so
    velocities to 1e-6 of their scale, positions to that and an ulp, and J to
    the 1e-6 of its FP32 summation order plus as much for the weights."""
    static, dyn = workloads.make_parameters(n, wind=wind, cfl=0.5, pbc=pbc)
    vth = 0.1                             # under C = 1 for every draw
    specs = [workloads.SpeciesSpec(24, weight=1e-3, vth=(vth,) * 3),
             workloads.SpeciesSpec(7, charge=1.0, mass=20.0, weight=3e-3, vth=(0.15, 0.05, 0.05),
                                   update_x=not frozen, update_u=not frozen)]
    parts, cfg = workloads.plasma(static, dyn, specs, seed=11)
    if frozen:
        cfg.update_x[1] = [True, False, True]
        cfg.update_u[1] = [False, True, True]
    p = oracle_params(static, dyn)
    fields = workloads.empty_fields(static, dyn)
    F = [gpu_field(random_field(p, 60 + c, scale=0.05)) for c in range(12)]
    fields = (tuple(F[:3]), tuple(F[3:6])) + fields[2:5] + ((tuple(F[6:9]), tuple(F[9:])),) + fields[6:]
    r = ElectrodynamicRunner(parts, cfg, fields, static, dyn, sort_every=0, tile=tile, rounds=4, min_blocks=4)
    assert not bool(N.lib().pic_tile_exact_grid(r.desc))
    for _ in range(4):                    # drift without a re-sort
        r.step()
    k = r.cur
    idx = torch.nonzero(r.act[k].view(-1)).view(-1)[::29]
    for a in range(3):                    # some particles within rounding of a face
        x = r.pos[k][a].view(-1)
        org, sp = float(r.desc.org_c[a]), float(r.desc.sp_c[a])
        x[idx] = (torch.floor((x[idx].double() - org) / sp) * sp + org).float()
    J1, x1, u1, a1, nr1 = _launch(r, False)
    J0, x0, u0, a0, nr0 = _launch(r, True)
    assert nr1 == -7 and 0 < nr0 <= a0.numel()
    assert torch.equal(a0, a1)
    for a in range(3):
        assert float((x0[a] - x1[a]).abs().max()) <= 1e-6 * wind[a]
    assert float((u0 - u1).abs().max()) <= 1e-6 * float(u1.abs().max())
    assert float((J0 - J1).norm() / J1.norm()) <= 2e-6


@pytest.mark.parametrize("tile", [4, 8])
@pytest.mark.parametrize("n,wind,pbc,frozen", [
    ((13, 10, 9), (1.3, 0.7, 2.1), (0, 0, 0), False),
    ((8, 8, 8), (0.9, 0.3, 1.1), (0, 1, 2), False),
    ((5, 4, 17), (0.1, 0.6, 1.9), (2, 0, 1), True),
])
def test_general_grid_direct_kernel_agrees_with_separate_kernels(tile, n, wind, pbc, frozen):
    """As above for the direct branch: push, half advance, boundaries, deposit,
    half advance, boundaries as separate launches, J in its own FP32 order."""
    static, dyn = workloads.make_parameters(n, wind=wind, cfl=0.5, pbc=pbc, current_deposition="direct")
    specs = [workloads.SpeciesSpec(24, weight=1e-3, vth=(0.1,) * 3),
             workloads.SpeciesSpec(7, charge=1.0, mass=20.0, weight=3e-3, vth=(0.15, 0.05, 0.05),
                                   update_x=not frozen, update_u=not frozen)]
    parts, cfg = workloads.plasma(static, dyn, specs, seed=12)
    if frozen:
        cfg.update_x[1] = [True, False, True]
        cfg.update_u[1] = [False, True, True]
    p = oracle_params(static, dyn)
    fields = workloads.empty_fields(static, dyn)
    F = [gpu_field(random_field(p, 80 + c, scale=0.05)) for c in range(12)]
    fields = (tuple(F[:3]), tuple(F[3:6])) + fields[2:5] + ((tuple(F[6:9]), tuple(F[9:])),) + fields[6:]
    r = ElectrodynamicRunner(parts, cfg, fields, static, dyn, sort_every=0, tile=tile)
    assert r.direct_general and not r.direct_fused and not r.defer_permute
    for _ in range(4):
        r.step()
    src, dst = r.cur, 1 - r.cur
    s = N.stream_handle()
    uo = [r.vel[dst][a] for a in range(3)]
    xd = [r.pos[dst][a] for a in range(3)]
    N.call("pic_push", r.desc, r.sp, r._pp(src), N.p3(r.E[r.ecur]), N.p3(r.B), r.Ee, r.Be, N.p3(uo), s)
    r.act[dst].copy_(r.act[src])
    half = pic_particles([r.pos[src][a] for a in range(3)], uo, r.act[dst])
    N.call("pic_advance_positions", r.desc, r.sp, half, 0.5, N.p3(xd), s)
    N.call("pic_particle_boundaries", r.desc, r.sp, r._pp(dst), s)
    for c in r.J:
        c.zero_()
    N.call("pic_deposit_direct", r.desc, r.sp, r._pp(dst), N.p3(r.J), s)
    N.call("pic_advance_positions", r.desc, r.sp, r._pp(dst), 0.5, N.p3(xd), s)
    N.call("pic_particle_boundaries", r.desc, r.sp, r._pp(dst), s)
    J1, x1, u1, a1 = torch.stack(r.J).clone(), r.pos[dst].clone(), r.vel[dst].clone(), r.act[dst].clone()
    for c in r.J:
        c.zero_()
    r.tile_ws[0] = -7
    N.call("pic_fused_push_direct_tiled_general", r.desc, r.sp, r._pp(src), N.p3(r.E[r.ecur]), N.p3(r.B), r.Ee,
           r.Be, r._pp(dst), N.p3(r.J), r.tile, N.ptr(r.starts), N.ptr(r.tile_ws), s)
    torch.cuda.synchronize()
    J0, x0, u0, a0 = torch.stack(r.J), r.pos[dst], r.vel[dst], r.act[dst]
    assert 0 <= int(r.tile_ws[0]) <= a0.numel()
    assert torch.equal(a0, a1)
    act = a0.view(r.S, r.P).unsqueeze(0).expand_as(x0)
    for a in range(3):
        assert float((x0[a] - x1[a]).abs()[act[a]].max()) <= 1e-6 * wind[a]
    assert float((u0 - u1).abs()[act].max()) <= 2e-6 * float(u1.abs().max())
    assert float((J0 - J1).norm() / J1.norm()) <= 2e-6
