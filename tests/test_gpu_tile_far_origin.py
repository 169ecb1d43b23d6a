"""Exact grids millions of spacings from the origin (through the C entry points;
the package's own grids are centred): the gathered Esirkepov launch reads
through its permutation and the direct launches run, as on a near grid.  A
shift of 5e6 keeps every node and half node an FP32 number; positions are
rounded to half cells, the FP32 spacing there."""

import numpy as np
import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import pic_particles
from pypic3d_amd.runner import ElectrodynamicRunner
from tests.gpu_helpers import gpu_field, oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu

SHIFT = 5.0e6


def _far_runner(current):
    static, dyn = workloads.make_parameters((20, 16, 12), wind=(20.0, 16.0, 12.0), cfl=0.5,
                                            current_deposition=current)
    specs = [workloads.SpeciesSpec(20, weight=0.01, vth=(0.12,) * 3),
             workloads.SpeciesSpec(6, charge=1.0, mass=20.0, weight=0.03, vth=(0.05,) * 3)]
    parts, cfg = workloads.plasma(static, dyn, specs, seed=5)
    p = oracle_params(static, dyn)
    f = [gpu_field(random_field(p, 70 + c, scale=0.05)) for c in range(6)]
    fields = (tuple(f[:3]), tuple(f[3:])) + workloads.empty_fields(static, dyn)[2:]
    r = ElectrodynamicRunner(parts, cfg, fields, static, dyn, sort_every=0, tile=4)
    assert r._pending and bool(N.lib().pic_tile_exact_grid(r.desc))
    x = r.pos[r._cur][0]                       # the permutation and the tiles are those of the unshifted cells
    x.copy_(torch.floor(2 * x) / 2 + SHIFT)
    r.desc.org_c[0] += SHIFT
    r.desc.org_v[0] += SHIFT
    r.desc.wind[0] = float(1 << 25)            # no wrap along x
    assert bool(N.lib().pic_tile_exact_grid(r.desc))
    return r


def _result(r, dst, nr):
    torch.cuda.synchronize()
    return torch.stack(r.J).clone(), r.pos[dst].clone(), r.vel[dst].clone(), r.act[dst].clone(), nr


def _launch(r, name, src, dst, *tail, perm=None, variant=0):
    for c in r.J:
        c.zero_()
    r.tile_ws[0] = -7
    r.desc.variant = variant
    first = (N.ptr(r.perm),) if perm else ()
    N.call(name, r.desc, r.sp, r._pp(src), *first, N.p3(r.E[r.ecur]), N.p3(r.B), r.Ee, r.Be, r._pp(dst), N.p3(r.J),
           r.tile, N.ptr(r.starts), *tail, N.ptr(r.tile_ws), N.stream_handle())
    r.desc.variant = 0
    return _result(r, dst, int(r.tile_ws[0]))


def _same(a, b):
    for q in (1, 2, 3):
        assert torch.equal(a[q], b[q])
    assert float((a[0] - b[0]).norm()) <= 1e-6 * float(b[0].norm()) and float(b[0].norm()) > 0


def test_gathered_esirkepov_launch_reads_through_the_permutation():
    r = _far_runner("esirkepov")
    src = r._cur
    a = _launch(r, "pic_fused_push_esirkepov_tiled_gather", src, 1 - src, 4, 4, perm=True)
    src = r.cur                                # applies the permutation
    strided = _launch(r, "pic_fused_push_esirkepov_tiled", src, 1 - src, 4, 4, variant=1)
    assert a[4] >= 0 and strided[4] == -7      # the tile kernel, not the strided one
    _same(a, strided)
    _same(_launch(r, "pic_fused_push_esirkepov_tiled", src, 1 - src, 4, 4), strided)


def test_direct_launches_run():
    r = _far_runner("j_from_rhov")
    assert r.direct_fused
    src = r._cur
    a = _launch(r, "pic_fused_push_direct_tiled_gather", src, 1 - src, 4, perm=True)
    src = r.cur
    dst = 1 - src
    _same(a, _launch(r, "pic_fused_push_direct_tiled", src, dst, 4))
    # the separate kernels, whose pushes round an ulp apart
    d, s = r.desc, N.stream_handle()
    for c in r.J:
        c.zero_()
    uo, xd = [r.vel[dst][c] for c in range(3)], [r.pos[dst][c] for c in range(3)]
    N.call("pic_push", d, r.sp, r._pp(src), N.p3(r.E[r.ecur]), N.p3(r.B), r.Ee, r.Be, N.p3(uo), s)
    r.act[dst].copy_(r.act[src])
    half = pic_particles([r.pos[src][c] for c in range(3)], uo, r.act[dst])
    N.call("pic_advance_positions", d, r.sp, half, 0.5, N.p3(xd), s)
    N.call("pic_particle_boundaries", d, r.sp, r._pp(dst), s)
    N.call("pic_deposit_direct", d, r.sp, r._pp(dst), N.p3(r.J), s)
    b = _result(r, dst, 0)
    assert float((a[2] - b[2]).abs().max()) <= 1e-6
    assert float((a[0] - b[0]).norm()) <= 1e-5 * float(b[0].norm())
