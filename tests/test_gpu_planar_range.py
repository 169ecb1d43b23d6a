"""The 1-D particle phase where cell indices are large: chunks of particles past
a million cells on the longest axes it takes, a chunk that spans such an axis,
and particles millions of cells outside a short domain.  FP32 step against the
FP64 kernels on the same FP32 inputs, in the cells the reference's modulo gives."""

import numpy as np
import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd._tensors import tiled_particles_from_arrays
from pypic3d_amd.evolve import time_loop_electrodynamic
from pypic3d_amd.particles.particle_class import SpeciesConfig

pytestmark = pytest.mark.gpu


def _positions(where, n, P, rng):
    if where == "upper end":
        c = np.sort(rng.integers(1_020_000, n - 3, P))
    elif where == "whole axis":
        c = np.sort(rng.integers(3, n - 3, P))
    else:                                           # either side of the domain, beyond what an estimate tells apart
        c = np.sort(rng.integers(4_300_000, 4_300_200, P)) * np.where(np.arange(P) < P // 2, -1, 1)
    return (c + rng.uniform(0.25, 0.75, P)) - n / 2


@pytest.mark.parametrize("where,n,spacing,P", [
    ("upper end", 1_040_000, 1.0, 700), ("upper end", 1_040_000, 0.1, 700), ("upper end", 1_040_000, 1.0, 1_050_000),
    ("whole axis", 1_040_000, 0.1, 700), ("outside", 64, 1.0, 700),
])
def test_large_cell_indices(where, n, spacing, P):
    """As in test_gpu_planar.py: velocities within 4e-6 of their scale, J within 1e-5 in the norm."""
    static, dyn = workloads.make_parameters((n, 1, 1), d=(spacing,) * 3, dt=0.2 * spacing)
    rng = np.random.default_rng(P)
    x = np.zeros((1, P, 3))
    x[0, :, 0] = _positions(where, n, P, rng) * spacing
    x = x.astype(np.float32).astype(np.float64)
    u = rng.uniform(-0.3, 0.3, (1, P, 3)).astype(np.float32).astype(np.float64)
    cfg = SpeciesConfig(charge=np.array([-1.0]), mass=np.array([1.0]), weight=np.array([0.1]),
                        update_x=np.ones((1, 3), bool), update_u=np.ones((1, 3), bool))
    gen = torch.Generator(device="cuda").manual_seed(5)
    EB = None

    def run(dtype):
        nonlocal EB
        f = workloads.empty_fields(static, dyn, dtype=dtype)
        if EB is None:
            EB = [torch.randn(f[0][0].shape, generator=gen, device="cuda") * 0.05 for _ in range(6)]
        f = (tuple(c.to(dtype) for c in EB[:3]), tuple(c.to(dtype) for c in EB[3:])) + f[2:]
        q, g = time_loop_electrodynamic(tiled_particles_from_arrays(x, u, np.ones((1, P), bool), dtype=dtype), cfg, f,
                                        static, dyn)
        return q.u.reshape(-1, 3).double(), [c.double() for c in g[2]]

    u0, J0 = run(torch.float32)
    u1, J1 = run(torch.float64)
    assert float((u0 - u1).abs().max()) <= 4e-6
    for a, b in zip(J0, J1):
        assert float((a - b).norm()) <= 1e-5 * float(b.norm())
