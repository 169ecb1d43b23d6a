"""The tile launches refuse what one launch cannot hold: 2^32 threads, which a
tile of 4^3 cells reaches on 1024^3 cells.  The refusal comes before anything
is launched, so the planes here are addresses that nothing reads."""

import numpy as np
import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc, make_species
from pypic3d_amd.particles.particle_class import SpeciesConfig


@pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are not memory")
@pytest.mark.parametrize("current,name,tail", [
    ("esirkepov", "pic_fused_push_esirkepov_tiled", (4, 4)),
    ("esirkepov", "pic_fused_push_esirkepov_tiled_general", (4,)),
    ("j_from_rhov", "pic_fused_push_direct_tiled", (4,)),
    ("j_from_rhov", "pic_fused_push_direct_tiled_general", ()),
])
def test_tile_launch_of_2_to_the_32_threads_is_refused(current, name, tail):
    N.load()
    static, dyn = workloads.make_parameters((1024,) * 3, d=(1.0,) * 3, dt=0.05, current_deposition=current)
    desc = make_desc(static, dyn)
    one = np.ones(1)
    sp = make_species(SpeciesConfig(one, one, one, np.ones((1, 3), bool), np.ones((1, 3), bool)), 1 << 20)
    at = iter(range(4096, 1 << 20, 4096))
    p3 = lambda: N.P3(*[next(at) for _ in range(3)])   # noqa: E731

    def particles():
        p = N.PicParticles()
        for a in range(3):
            p.x[a], p.u[a] = next(at), next(at)
        p.active = next(at)
        return p

    with pytest.raises(ValueError):
        N.call(name, desc, sp, particles(), p3(), p3(), None, None, particles(), p3(), 4, N.c_vp(next(at)), *tail,
               N.c_vp(next(at)), None)
