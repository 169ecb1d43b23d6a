"""Guard refresh and conducting walls of 2-D grids whose planes have more than
2^28 rows of one cell (a launch of 64 threads a row in one grid axis would pass
2^32 threads), and with more than 2^31 guard cells (numbered in 64 bits)."""

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc

pytestmark = pytest.mark.gpu

SIDE = 16400        # (SIDE + 2)^2 and SIDE^2 > 2^28


def _field(desc, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(tuple(desc.dims), generator=gen, device="cuda") + 1.0


@pytest.mark.parametrize("side,g", [(SIDE, 1), (23200, 2)])
def test_refresh_of_a_wide_plane(side, g):
    static, dyn = workloads.make_parameters((side, side, 1), dt=0.05, g=g)
    desc = make_desc(static, dyn)
    f = _field(desc, 1)
    inner = f[g:-g, g:-g, g].clone()
    N.call("pic_halo_refresh", desc, N.ptr(f), 0, N.stream_handle())
    rows = torch.cat([inner[-g:], inner, inner[:g]])
    want = torch.cat([rows[:, -g:], rows, rows[:, :g]], dim=1)
    for k in range(2 * g + 1):
        assert torch.equal(f[:, :, k], want)


def test_walls_of_a_wide_plane():
    static, dyn = workloads.make_parameters((SIDE, SIDE, 1), dt=0.05, g=1, bc=(1, 0, 0))
    desc = make_desc(static, dyn)
    E = [_field(desc, c) for c in range(3)]
    want = [c[2:-2, 1:-1, 1].clone() for c in E]
    first = E[0][1, 1:-1, 1].clone()
    N.call("pic_conducting_walls", desc, N.p3(E), N.stream_handle())
    for c in range(3):
        assert torch.equal(E[c][2:-2, 1:-1, 1], want[c])
        for plane in (1, -2):
            assert bool((E[c][plane, 1:-1, 1] == 0).all()) == (c != 0)
    assert torch.equal(E[0][1, 1:-1, 1], first)
