"""Tile kernels with few and many slots per tile (one, two and four consecutive slots per thread) and with slots
that no tile holds, shared out over blocks, against the slot-ordered kernels on the same particles."""

import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd._tensors import soa_view
from pypic3d_amd.particles.particle_class import TiledParticles
from pypic3d_amd.runner import ElectrodynamicRunner
from tests.gpu_helpers import gpu_field, oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu


# 4^3-cell tiles: a mean of up to 256 slots takes one slot per thread, up to 512 two, more than that four
@pytest.mark.parametrize("current", ["esirkepov", "j_from_rhov"])
@pytest.mark.parametrize("wind", [(13.0, 9.0, 10.0), (1.3, 0.7, 2.1)])      # FP32 node lines, and not
@pytest.mark.parametrize("ppc,empty", [(1, 0), (4, 1), (4, 3000), (9, 517), (24, 131), (30, 60000)])
def test_steps_on_tiles_agree_with_slot_order(ppc, empty, wind, current):
    """Particle outputs to FP32 rounding of positions and pushes, fields and J to the FP32 summation order."""
    n = (13, 9, 10)
    static, dyn = workloads.make_parameters(n, wind=wind, cfl=0.5, current_deposition=current)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(ppc, weight=1e-3, vth=(0.1,) * 3),
                                                workloads.SpeciesSpec(ppc, charge=1.0, mass=9.0, weight=1e-3,
                                                                      vth=(0.05,) * 3)], seed=ppc)
    x, u = parts.x[0, 0, 0], parts.u[0, 0, 0]                     # (S, P, 3)
    S, P = x.shape[:2]
    grow = lambda t: torch.cat([t, torch.full((S, empty, 3), 0.1, device=t.device)], 1).permute(2, 0, 1).contiguous()   # noqa: E731
    act = torch.cat([parts.active.view(S, P), torch.zeros((S, empty), dtype=torch.bool, device=x.device)], 1)
    order = torch.randperm(P + empty, generator=torch.Generator().manual_seed(7)).to(x.device)
    x, u, act = grow(x)[:, :, order].contiguous(), grow(u)[:, :, order].contiguous(), act[:, order].contiguous()
    p = oracle_params(static, dyn)
    F = [gpu_field(random_field(p, 30 + c, scale=0.02)) for c in range(6)]
    got = []
    for tile in (4, None):
        fields = workloads.empty_fields(static, dyn)
        fields = (tuple(f.clone() for f in F[:3]), tuple(f.clone() for f in F[3:])) + tuple(fields[2:])
        pp = TiledParticles(soa_view(x.clone()), soa_view(u.clone()), act.clone().view(1, 1, 1, S, P + empty))
        r = ElectrodynamicRunner(pp, cfg, fields, static, dyn, sort_every=0, tile=tile)
        for _ in range(2):
            r.step()
        torch.cuda.synchronize()
        out, f = r.state()
        on = out.active.view(-1)
        assert int(on.sum()) == int(act.sum())
        q = torch.cat([out.x.reshape(-1, 3), out.u.reshape(-1, 3)], 1)[on].double()
        assert float(torch.cat([out.x.reshape(-1, 3), out.u.reshape(-1, 3)], 1)[~on].abs().sum()) == 0.0
        got.append((q.sum(0), q.square().sum(0), [torch.stack(list(c)).double() for c in f[:3]]))
    (s1, v1, f1), (s0, v0, f0) = got
    scale = torch.sqrt(v0 * int(act.sum()))
    # a sum over particles that differ by FP32 rounding; one that rounds across a periodic face moves by the box,
    # which the squares do not see
    assert float(((s1 - s0).abs() / scale)[3:].max()) <= 1e-5
    assert float(((v1 - v0).abs() / v0).max()) <= 1e-5
    for a, b in zip(f1, f0):
        assert float((a - b).norm() / b.norm()) <= 1e-5
