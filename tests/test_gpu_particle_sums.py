"""Kinetic energy and momentum of slots read four at a time and singly: species that end inside a group of four,
remainders, planes off 16 bytes, more slots than one round of the grid, empty slots, speeds from rest to near c."""

import numpy as np
import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd._tensors import tiled_particles_from_arrays
from pypic3d_amd.particles.particle_class import SpeciesConfig
from pypic3d_amd.utils import compute_energy, compute_total_momentum

pytestmark = pytest.mark.gpu


# planes start on 16 bytes where count * slots is a multiple of 4
@pytest.mark.parametrize("count,slots", [(1, 1), (1, 3), (1, 4), (2, 2), (4, 5), (4, 1), (3, 7), (2, 1026), (16, 33),
                                         (1, 1 << 21), (1, (1 << 20) + 3)])
def test_kinetic_energy_and_momentum(count, slots):
    static, dyn = workloads.make_parameters((6, 5, 4), cfl=0.5)
    C = float(dyn.C)
    rng = np.random.default_rng(count * 1000 + slots)
    u = (rng.standard_normal((count, slots, 3)) * 0.1).clip(-0.5, 0.5)
    u[:, ::3] *= 1e-6
    u[:, 1::5] = np.array([0.577, -0.577, 0.577])     # 0.9994 c
    u[:, 2::7] = 0.0
    u = (u * C).astype(np.float32)
    act = rng.random((count, slots)) < 0.9
    mass, weight = 1.0 + np.arange(count), 0.5 + 0.25 * np.arange(count)
    free = np.ones((count, 3), bool)
    cfg = SpeciesConfig(-np.ones(count), mass, weight, free, free)
    parts = tiled_particles_from_arrays(np.zeros_like(u), u, act)
    fields = workloads.empty_fields(static, dyn)
    kinetic = float(compute_energy(parts, fields[0], fields[1], static, dyn, cfg)[2])
    momentum = float(compute_total_momentum(parts, cfg))
    v2 = (u.astype(np.float64) ** 2).sum(-1)
    mw = (mass * weight)[:, None] * act
    r = np.sqrt(1.0 - v2 / C ** 2)
    # per term a few roundings of 1.1e-16, times 1 / r^2 = 1000 for those next to 1 in 1 - v^2/C^2
    assert kinetic == pytest.approx(float((mw * v2 / (r * (1.0 + r))).sum()), rel=1e-12)
    assert momentum == pytest.approx(float((mw * np.sqrt(v2)).sum()), rel=1e-13)
