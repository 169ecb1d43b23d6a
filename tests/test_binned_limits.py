"""The workspace query of the binned deposits is the rule by which a call takes
them: it refuses every set their entry points refuse (host code, no GPU)."""

import numpy as np
import pytest

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc, make_species
from pypic3d_amd.particles.particle_class import SpeciesConfig

LIMIT = 2 ** 31 - 2048      # slots, numbered in 32 bits with room for a block's overhang


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_sets_beyond_32_bit_slots_are_not_binned(kind):
    import torch  # noqa: F401  (load order: torch's HIP runtime first)
    static, dyn = workloads.make_parameters((64, 64, 64), dt=0.05)
    desc = make_desc(static, dyn)

    def query(count, slots):
        one = np.ones(count)
        cfg = SpeciesConfig(one, one, one, np.ones((count, 3), bool), np.ones((count, 3), bool))
        return int(N.load().pic_binned_workspace_bytes(desc, make_species(cfg, slots), kind))

    record = 16 if kind == 0 else 32
    assert query(1, LIMIT - 1) > record * (LIMIT - 1)
    assert query(2, LIMIT // 2 - 1) > record * (LIMIT - 2)
    for count, slots in ((1, LIMIT), (1, 2 ** 31 - 1), (2, LIMIT // 2), (2, 2 ** 30), (16, 2 ** 31 - 1)):
        assert query(count, slots) == -1
