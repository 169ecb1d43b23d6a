"""Face crossings beyond what a work item's queue holds (pic_binned.hip): most
particles of an 8^3 tile leave their cell, so an item of eight passes empties
its queue several times.  The raw deposit against the FP64 oracle, with the
parity tolerance of the FP32 kernels: a particle dropped or deposited twice
changes J by some 1e-2 of its largest value."""

import numpy as np
import pytest
import torch

from oracle import pic_oracle as O
from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc, make_species, particle_planes, pic_particles, tiled_particles_from_arrays
from pypic3d_amd.particles.particle_class import SpeciesConfig
from tests.gpu_helpers import TOL, host, oracle_params, rel_err
from tests.helpers import random_particles, species

pytestmark = pytest.mark.gpu


# vmax in cells a step and axis.  Of the passes' 1024 particles 0.97 queues some 870 (emptied after every second
# pass), 0.4 some 500 (after every third), 0.15 some 210 (after the fifth and the last).
@pytest.mark.parametrize("spacing", [0.5, 0.3])
@pytest.mark.parametrize("vmax", [0.97, 0.4, 0.15])
@pytest.mark.parametrize("P", [8192, 20011])
def test_deposit_of_more_crossings_than_the_queue_holds(spacing, vmax, P):
    static, dyn = workloads.make_parameters((8, 8, 8), d=(spacing,) * 3, dt=0.05)
    p = oracle_params(static, dyn)
    x, u, act = random_particles(p, S=2, P=P, seed=P, vmax=vmax, inactive_frac=0.01)
    sp = species(2, charge=(-1.0, 2.0), mass=(1.0, 50.0), weight=(0.5, 0.25))
    cfg = SpeciesConfig(sp.charge, sp.mass, sp.weight, sp.update_x, sp.update_u)
    desc, csp = make_desc(static, dyn), make_species(cfg, P)
    parts = tiled_particles_from_arrays(x, u, act)
    J = [torch.zeros(p.shape, dtype=torch.float32, device="cuda") for _ in range(3)]
    ws = torch.empty(int(N.lib().pic_binned_workspace_bytes(desc, csp, 2)), dtype=torch.uint8, device="cuda")
    N.call("pic_deposit_esirkepov_binned", desc, csp, pic_particles(*particle_planes(parts)), N.p3(J), N.ptr(ws),
           ws.numel(), N.stream_handle())
    for a, b in zip(J, O.esirkepov_raw(x, u, act, sp, p)):
        assert rel_err(host(a), b) <= TOL
