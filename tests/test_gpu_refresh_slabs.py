"""Guard refresh, whose threads number the guard cells slab by slab, bit for bit
against the oracle: both types, reduced and short axes, one guard cell and three,
and the zeros behind walls."""

import numpy as np
import pytest
import torch

from oracle import pic_oracle as O
from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc
from tests.gpu_helpers import oracle_params
from tests.helpers import random_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("bc", [(0, 0, 0), (1, 0, 2)])
@pytest.mark.parametrize("n,g", [((9, 7, 59), 2), ((2, 2, 2), 2), ((9, 1, 61), 2), ((70, 33, 1), 1), ((300, 1, 1), 3),
                                 ((5, 1, 57), 3), ((5, 1, 58), 3), ((1, 1, 63), 1), ((1, 600, 3), 2)])
def test_refresh_matches_the_oracle(n, g, bc, dtype):
    static, dyn = workloads.make_parameters(n, dt=0.05, g=g, bc=bc)
    p = oracle_params(static, dyn)
    f = random_field(p, 3, refresh=False)
    t = torch.tensor(f, dtype=dtype, device="cuda")
    N.call(N.op("pic_halo_refresh", dtype == torch.float64), make_desc(static, dyn), N.ptr(t), 0, N.stream_handle())
    np.testing.assert_array_equal(t.double().cpu().numpy(), O.refresh(f, p, bc))
