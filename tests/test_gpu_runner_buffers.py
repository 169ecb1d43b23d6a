"""The runner's current stays in its own arrays: a view taken from state() shows
the current of every later step, filter or none, tiles or none."""

import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd.runner import ElectrodynamicRunner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("current_filter", ["none", "bilinear", "digital"])
@pytest.mark.parametrize("spacing,tile", [(1.0, None), (1.0, 4), (0.1, 4), (1.0, 8)])
def test_views_of_the_current_stay_current(current_filter, spacing, tile):
    static, dyn = workloads.make_parameters((12, 16, 20), d=(spacing,) * 3, cfl=0.4, alpha=0.8,
                                            current_deposition="j_from_rhov", current_filter=current_filter)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(4, weight=0.01, vth=(0.1,) * 3)], seed=2)
    r = ElectrodynamicRunner(parts, cfg, workloads.empty_fields(static, dyn), static, dyn, sort_every=2, tile=tile)
    J = r.state()[1][2]
    at = [c.data_ptr() for c in J]
    for _ in range(3):
        before = [c.clone() for c in J]
        r.step()
        assert [c.data_ptr() for c in r.state()[1][2]] == at == [c.data_ptr() for c in r.J]
        for a, b in zip(J, before):
            assert float(a.abs().max()) > 0 and not torch.equal(a, b)


@pytest.mark.parametrize("current", ["esirkepov", "j_from_rhov"])
@pytest.mark.parametrize("tile", [None, 4])
@pytest.mark.parametrize("current_filter", ["none", "digital"])
def test_steps_allocate_nothing(current, tile, current_filter):
    static, dyn = workloads.make_parameters((16, 16, 20), d=(1.0,) * 3, cfl=0.4, alpha=0.8,
                                            current_deposition=current, current_filter=current_filter)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(8, weight=0.01, vth=(0.1,) * 3)], seed=2)
    r = ElectrodynamicRunner(parts, cfg, workloads.empty_fields(static, dyn), static, dyn, sort_every=2, tile=tile)
    assert r.S * r.P >= 1 << 15             # the deposit in any order takes a workspace from here on
    for _ in range(2):                      # the buffers of the first step and the first re-sort
        r.step()
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]   # noqa: E731
    before = count()
    for _ in range(4):
        r.step()
    assert count() == before
