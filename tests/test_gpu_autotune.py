"""The runner's autotune launches the entry point its steps launch, and every
candidate shape where the kernel that runs has several."""

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd.runner import ElectrodynamicRunner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spacing,variant,name,shapes", [
    (1.0, 0, "pic_fused_push_esirkepov_tiled", 1),
    (0.1, 0, "pic_fused_push_esirkepov_tiled_general", 1),
    (1.0, 1, "pic_fused_push_esirkepov_tiled", 9),
    (0.1, 1, "pic_fused_push_esirkepov_tiled", 9),
])
def test_tile_autotune_times_the_kernel_of_the_steps(monkeypatch, spacing, variant, name, shapes):
    static, dyn = workloads.make_parameters((12, 16, 8), d=(spacing,) * 3, cfl=0.4)
    parts, cfg = workloads.plasma(static, dyn, [workloads.SpeciesSpec(4, weight=0.01, vth=(0.1,) * 3)], seed=2)
    r = ElectrodynamicRunner(parts, cfg, workloads.empty_fields(static, dyn), static, dyn, sort_every=0, tile=4)
    r.cur
    r.desc.variant = variant
    seen = []
    call = N.call
    monkeypatch.setattr(N, "call", lambda n, *a: (seen.append(n), call(n, *a))[1])
    best, times = r.autotune(reps=2)
    tuned = set(seen)
    seen.clear()
    r.step()
    assert tuned == {name} == {n for n in seen if n.startswith("pic_fused")}
    assert len(times) == shapes and f"{best[0]}/{best[1]}" in times and best == (r.rounds, r.min_blocks)
