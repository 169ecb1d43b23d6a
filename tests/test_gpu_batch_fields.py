"""The ensemble's field passes against the single-simulation kernels on the same
arrays: few members (many blocks each) and more than a pass has blocks, 1-D, 2-D
and 3-D members mixed, axes as short as the guard band, one and three guard
cells, and currents in every guard cell."""

import ctypes

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc
from pypic3d_amd.batch import PicBatchSim
from pypic3d_amd.deposition.Esirkepov import finish_current
from pypic3d_amd.solvers.first_order_yee import yee_b, yee_e

pytestmark = pytest.mark.gpu

SHAPES = [(64, 1, 1), (33, 21, 1), (7, 9, 5), (1, 6, 12), (3, 3, 1), (3, 1, 50)]


@pytest.mark.parametrize("members,g", [(1, 2), (7, 2), (6, 1), (6, 3), (1300, 2)])
def test_field_step_matches_the_single_simulation_kernels(members, g):
    """The same expressions point by point: a few FP32 roundings apart at most."""
    table = (PicBatchSim * members)()
    descs, off, at = [], 0, []
    for m in range(members):
        static, dyn = workloads.make_parameters(SHAPES[m % len(SHAPES)], cfl=0.4, g=g)
        d = make_desc(static, dyn)
        ctypes.memmove(ctypes.addressof(table[m].desc), ctypes.addressof(d), ctypes.sizeof(N.PicDesc))
        table[m].species.count = 1
        table[m].field_offset = off
        descs.append(d)
        at.append(off)
        off += d.dims[0] * d.dims[1] * d.dims[2]
    N.check(N.lib().pic_batch_check(ctypes.addressof(table), members, 0, off), "pic_batch_check")
    gen = torch.Generator(device="cuda").manual_seed(members + g)
    F = {k: torch.randn((3, off), generator=gen, device="cuda") for k in ("E", "B", "J")}
    single = {k: v.clone() for k, v in F.items()}
    tab = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    Bh, Eo = torch.full_like(F["B"], 7.0), torch.full_like(F["E"], 7.0)
    s = N.stream_handle()
    N.call("pic_batch_field_step", tab.data_ptr(), members, N.p3(F["E"]), N.p3(F["B"]), N.p3(Bh), N.p3(F["J"]),
           N.p3(Eo), s)
    for m in sorted({0, members // 2, members - 1, *range(min(members, 6))}):
        d, shape = descs[m], tuple(descs[m].dims)
        n = shape[0] * shape[1] * shape[2]
        E, B, J = ([single[k][c, at[m]:at[m] + n].clone().view(shape) for c in range(3)] for k in ("E", "B", "J"))
        B1, E1, B2 = ([torch.empty_like(c) for c in E] for _ in range(3))
        finish_current(d, J, s)
        yee_b(d, E, B, B1, False, s)
        yee_e(d, E, B1, J, E1, s)
        yee_b(d, E1, B1, B2, False, s)
        for got, want in ((F["J"], J), (Bh, B1), (Eo, E1), (F["B"], B2)):
            for c in range(3):
                a = got[c, at[m]:at[m] + n].view(shape)
                assert float((a - want[c]).abs().max()) <= 4e-6 * float(want[c].abs().max())


def test_more_work_items_than_one_launch_holds():
    """A block per item would pass 2^32 threads at 2^23 items.  Member 1's only
    item stands last, behind that many of member 0's (which repeat its step)."""
    members, slots = 2, 300
    static, dyn = workloads.make_parameters((8, 1, 1), dt=0.05)
    d = make_desc(static, dyn)
    table = (PicBatchSim * members)()
    cells = d.dims[0] * d.dims[1] * d.dims[2]
    for m in range(members):
        ctypes.memmove(ctypes.addressof(table[m].desc), ctypes.addressof(d), ctypes.sizeof(N.PicDesc))
        sp = table[m].species
        sp.count, sp.slots = 1, slots
        sp.charge[0], sp.mass[0], sp.weight[0] = -1.0, 1.0, 0.01
        for a in range(3):
            sp.update_x[0][a] = sp.update_u[0][a] = 1
        table[m].particle_offset, table[m].field_offset = m * slots, m * cells
    N.check(N.lib().pic_batch_check(ctypes.addressof(table), members, 2 * slots, 2 * cells), "pic_batch_check")
    tab = torch.frombuffer(bytearray(bytes(table)), dtype=torch.uint8).cuda()
    work = torch.zeros(((1 << 23) + 2, 2), dtype=torch.int32, device="cuda")
    work[-1, 0] = 1
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = (torch.rand((3, 2 * slots), generator=gen, device="cuda") - 0.5) * 0.5
    u = (torch.rand((3, 2 * slots), generator=gen, device="cuda") - 0.5) * 0.2
    act = torch.ones(2 * slots, dtype=torch.uint8, device="cuda")
    E, B, J = (torch.zeros((3, 2 * cells), device="cuda") for _ in range(3))
    xo, uo, ao = torch.full_like(x, 9.0), torch.full_like(u, 9.0), torch.zeros_like(act)

    def planes(xs, us, a):
        p = N.PicParticles()
        for c in range(3):
            p.x[c], p.u[c] = xs[c].data_ptr(), us[c].data_ptr()
        p.active = a.data_ptr()
        return p

    N.call("pic_batch_fused_push_esirkepov", tab.data_ptr(), work.data_ptr(), work.shape[0], 2, 64, planes(x, u, act),
           N.p3(E), N.p3(B), planes(xo, uo, ao), N.p3(J), N.stream_handle())
    assert bool((ao == 1).all())
    assert float((uo - u).abs().max()) <= 1e-6 and float((xo - x - 0.05 * u).abs().max()) <= 1e-6
