"""Flags of non-zero external fields: first and last value, NaN, signed zeros, each component, both types."""

import pytest
import torch

from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [(1, 1, 3), (30, 21, 17), (130, 90, 70)])
def test_any_nonzero_flags(n, dtype):
    static, dyn = workloads.make_parameters(n, cfl=0.5)
    desc = make_desc(static, dyn)
    shape = tuple(m + 4 for m in n)
    a = [torch.zeros(shape, dtype=dtype, device="cuda") for _ in range(6)]
    flags = torch.full((2,), 7, dtype=torch.int32, device="cuda")

    def ask():
        N.call(N.op("pic_any_nonzero", dtype == torch.float64), desc, N.p3(a[:3]), N.p3(a[3:]), N.ptr(flags),
               N.stream_handle())
        return flags.tolist()
    a[1].view(-1)[3] = -0.0
    assert ask() == [0, 0]
    for c, where, value in ((0, 0, 1e-40), (2, -1, float("nan")), (3, -1, -2.0), (5, a[0].numel() // 2, float("inf"))):
        a[c].view(-1)[where] = value
        assert ask() == ([1, 0] if c < 3 else [0, 1])
        a[c].zero_()
    a[0].view(-1)[5] = a[4].view(-1)[6] = 1.0
    assert ask() == [1, 1]
