"""First-order 1-D and 2-D particle phase (chunks with field and current boxes in
LDS) against the separate FP64 kernels on the same FP32 inputs: grids whose
lines are no FP32 numbers, every particle boundary, frozen axes, slots in cell
order (boxed ranges) and shuffled (wider ranges), chunk and group remainders,
species that change inside a thread's group, steps longer than a cell."""

import numpy as np
import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd._tensors import tiled_particles_from_arrays
from pypic3d_amd.evolve import time_loop_electrodynamic
from pypic3d_amd.particles.particle_class import SpeciesConfig
from tests.gpu_helpers import gpu_field, oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu


def _case(n, wind, pbc, P, order, dt, ext, seed):
    static, dyn = workloads.make_parameters(n, wind=wind, cfl=0.4, dt=dt, pbc=pbc)
    p = oracle_params(static, dyn)
    rng = np.random.default_rng(seed)
    S = 3
    w, dd = np.array(wind), np.array(wind) / np.array(n)
    x = (rng.random((S, P, 3)) - 0.5) * w
    if order == "sorted":
        c = [np.clip(np.floor((x[..., a] + w[a] / 2) / dd[a]), 0, n[a] - 1) for a in range(3)]
        perm = np.argsort((c[0] * n[1] + c[1]) * n[2] + c[2], axis=1, kind="stable")
        x = np.take_along_axis(x, perm[..., None], 1)
    x = x.astype(np.float32).astype(np.float64)
    u = rng.normal(0, 0.1, (S, P, 3)) + np.array([0.2, -0.1, 0.05])
    u = (u / np.maximum(1.0, np.linalg.norm(u, axis=-1, keepdims=True) / 0.9)).astype(np.float32).astype(np.float64)
    act = rng.random((S, P)) < 0.95
    cfg = SpeciesConfig(charge=np.array([-1.0, 1.0, -1.0]), mass=np.array([1.0, 20.0, 2.0]),
                        weight=np.array([0.1, 0.1, 0.02]),
                        update_x=np.array([[True] * 3, [True] * 3, [True, False, True]]),
                        update_u=np.array([[True] * 3, [True] * 3, [False, True, True]]))
    f = [random_field(p, seed + c, scale=0.05 if c < 6 else 0.02).astype(np.float32).astype(np.float64)
         for c in range(12)]

    def run(dtype):
        parts = tiled_particles_from_arrays(x, u, act, dtype=dtype)
        fields = workloads.empty_fields(static, dyn, dtype=dtype)
        t = [gpu_field(a).to(dtype) for a in f]
        e = (tuple(t[6:9]), tuple(t[9:])) if ext else fields[5]
        fields = (tuple(t[:3]), tuple(t[3:6])) + fields[2:5] + (e,) + fields[6:]
        q, g = time_loop_electrodynamic(parts, cfg, fields, static, dyn)
        return (q.x.reshape(-1, 3).double(), q.u.reshape(-1, 3).double(), q.active.reshape(-1),
                torch.stack([c.double() for c in g[2]]))
    return run, act


@pytest.mark.parametrize("n,wind,pbc,P,order,dt,ext", [
    ((37, 1, 1), (3.7, 0.1, 0.1), (0, 0, 0), 1, "sorted", None, True),
    ((37, 1, 1), (3.7, 0.1, 0.1), (1, 0, 0), 257, "sorted", None, False),
    ((64, 1, 1), (64.0, 1.0, 1.0), (2, 0, 0), 1023, "shuffled", 2.7, True),
    ((4000, 1, 1), (390.0, 0.1, 0.1), (0, 0, 0), 5000, "shuffled", None, True),
    ((4000, 1, 1), (390.0, 0.1, 0.1), (0, 0, 0), 400001, "sorted", None, True),
    ((19, 13, 1), (1.9, 1.1, 0.1), (0, 0, 0), 255, "sorted", None, True),
    ((19, 13, 1), (1.9, 1.1, 0.1), (1, 2, 0), 3001, "shuffled", None, True),
    ((24, 40, 1), (24.0, 40.0, 1.0), (0, 0, 0), 2050, "sorted", 2.3, False),
    ((48, 40, 1), (4.7, 4.1, 0.1), (0, 0, 0), 4099, "shuffled", None, True),
    ((130, 70, 1), (13.1, 6.9, 0.1), (0, 0, 0), 3003, "shuffled", None, True),
    ((65, 33, 1), (6.5, 3.1, 0.1), (0, 1, 0), 400003, "sorted", None, True),
])
def test_planar_particle_phase_matches_fp64_kernels(n, wind, pbc, P, order, dt, ext):
    """Inputs are FP32 numbers in both runs.  FP32 weights, push and displacement
    put velocities within 4e-6 of their scale (five rounded square roots and
    reciprocals of 1 ulp among some twenty operations), positions within that times
    dt and an ulp of the domain, J within 1e-5 in the norm (terms of both signs)."""
    run, act = _case(n, wind, pbc, P, order, dt, ext, seed=sum(n) + P)
    x1, u1, a1, J1 = run(torch.float64)
    x0, u0, a0, J0 = run(torch.float32)
    step = dt if dt is not None else 0.4 * min(w / m for w, m in zip(wind, n))
    near = torch.zeros_like(a1)
    for a in range(3):      # an FP32 rounding may decide a wrap, a reflection or an absorption at the wall
        if n[a] > 1 or pbc[a] == 0:
            near |= (x1[:, a].abs() - wind[a] / 2).abs() <= 4e-6 * (wind[a] + step)
    assert bool((a0 == a1)[~near].all())
    ok = a0 & a1 & ~near
    assert int(ok.sum()) >= 0.5 * int((a0 & a1).sum())
    for a in range(3):
        assert float((x0[ok, a] - x1[ok, a]).abs().max()) <= 4e-6 * step + 2e-7 * wind[a]
    assert float((u0[ok] - u1[ok]).abs().max()) <= 4e-6
    assert float((J0 - J1).norm()) <= 1e-5 * float(J1.norm())
