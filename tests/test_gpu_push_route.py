"""Which sets the push takes through tiles, and that the two routes agree at the
line between them (same stencils, sums in another order: a few ulp of |v| <= 1)."""

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd.pusher.particle_push import particle_push
from tests.gpu_helpers import gpu_field, oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sf,ppc,tiles", [
    ((32, 32, 32), 1, 31, False), ((32, 32, 32), 1, 32, True), ((32, 32, 32), 2, 7, False), ((32, 32, 32), 2, 8, True),
    ((16, 16, 16), 2, 64, False), ((16, 16, 16), 2, 112, True), ((64, 64, 1), 1, 300, False),
])
def test_push_route(monkeypatch, n, sf, ppc, tiles):
    static, dyn = workloads.make_parameters(n, d=(0.5,) * 3, dt=0.05, shape_factor=sf)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(ppc, weight=0.01, vth=(0.1,) * 3)], seed=4)
    order = torch.randperm(parts.x.shape[4], device="cuda")
    parts = parts._replace(x=parts.x[..., order, :], u=parts.u[..., order, :])
    p = oracle_params(static, dyn)
    E, B = (tuple(gpu_field(random_field(p, s + c, scale=0.2)) for c in range(3)) for s in (1, 4))
    seen, call = [], N.call
    monkeypatch.setattr(N, "call", lambda name, *a: (seen.append(name), call(name, *a))[1])
    got = particle_push(parts, cfg, E, B, static, dyn).u
    assert ("pic_push_binned" in seen) == tiles and ("pic_push" in seen) != tiles
    monkeypatch.setattr("pypic3d_amd.pusher.particle_push._through_tiles", lambda d, s: not tiles)
    other = particle_push(parts, cfg, E, B, static, dyn).u
    assert float((got - other).abs().max()) <= 8 * 2.0 ** -23
