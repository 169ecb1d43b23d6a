"""Fold + refresh, filter + refresh (+ conducting walls) and the walls alone, each one launch for three components,
against the oracle's sequential fold, refresh, filter and wall operations: axes shorter than two guard bands,
reduced axes, every boundary code, FP32 and FP64."""

import numpy as np
import pytest
import torch

from oracle import pic_oracle as O
from pypic3d_amd import _native as N
from pypic3d_amd import workloads
from pypic3d_amd._tensors import make_desc
from tests.gpu_helpers import oracle_params

pytestmark = pytest.mark.gpu

SHAPES = [(9, 8, 70), (2, 3, 5), (12, 1, 1), (1, 6, 130), (4, 5, 1)]
CODES = [(0, 0, 0), (1, 0, 2), (2, 1, 0), (1, 1, 1)]


def _setup(shape, bc, pbc, alpha=1.0, g=2):
    static, dyn = workloads.make_parameters(shape, dt=0.05, bc=bc, pbc=pbc, alpha=alpha, g=g)
    p = oracle_params(static, dyn)
    rng = np.random.default_rng(7)
    f = [rng.standard_normal(p.shape).astype(np.float32).astype(np.float64) for _ in range(3)]
    return make_desc(static, dyn), p, f


def _gpu(f, dtype):
    return [torch.as_tensor(c, dtype=dtype, device="cuda").contiguous() for c in f]


def _close(got, want, dtype, terms):
    """terms values of order one are added: the rounding of a sum is below terms^2 eps of its largest value."""
    eps = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -53
    for a, b in zip(got, want):
        a = a.double().cpu().numpy()
        assert np.max(np.abs(a - b)) <= terms * terms * eps * max(1.0, np.max(np.abs(b)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("codes", CODES)
def test_finish_equals_fold_then_refresh(shape, codes, dtype):
    desc, p, f = _setup(shape, (0, 0, 0), codes)
    t = _gpu(f, dtype)
    N.call(N.op("pic_finish_current", dtype == torch.float64), desc, N.p3(t), 1, N.stream_handle())
    want = [O.refresh(O.fold(c, p, p.particle_bc), p, p.particle_bc) for c in f]
    _close(t, want, dtype, 125)      # two reduced axes: 25 cells and their images


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape,g", [(s, 2) for s in SHAPES] + [((6, 5, 7), 1), ((5, 6, 8), 3)])
@pytest.mark.parametrize("bc", [(0, 0, 0), (1, 0, 0), (1, 1, 1)])
@pytest.mark.parametrize("bilinear,walls", [(0, 0), (1, 0), (0, 1)])
def test_filter_refresh_equals_the_separate_operations(shape, g, bc, bilinear, walls, dtype):
    if any(1 < n < g for n in shape):
        pytest.skip("an axis narrower than the guard band is refused")
    desc, p, f = _setup(shape, bc, (0, 0, 0), alpha=0.7, g=g)
    f = [O.refresh(c, p) for c in f]
    src, out = _gpu(f, dtype), [torch.full(p.shape, 9.0, dtype=dtype, device="cuda") for _ in range(3)]
    N.call(N.op("pic_filter_refresh", dtype == torch.float64), desc, N.p3(src), N.p3(out), bilinear, 0.7, 0, walls,
           N.stream_handle())
    want = [O.bilinear_filter(c, p.g) if bilinear else O.digital_filter(c, 0.7, p.g) for c in f]
    if walls:
        for axis in range(3):
            want = [O.zero_boundary(c, p, axis) if i != axis else c for i, c in enumerate(want)]
    _close(out, [O.refresh(c, p) for c in want], dtype, 27)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bc", [(0, 0, 0), (1, 0, 0), (0, 1, 1), (1, 1, 1)])
def test_conducting_walls_zero_the_tangential_components(shape, bc, dtype):
    desc, p, f = _setup(shape, bc, (0, 0, 0))
    f = [O.refresh(c, p) for c in f]
    t = _gpu(f, dtype)
    N.call(N.op("pic_conducting_walls", dtype == torch.float64), desc, N.p3(t), N.stream_handle())
    for i, c in enumerate(f):
        for axis in range(3):
            if axis != i:
                c = O.zero_boundary(c, p, axis)
        np.testing.assert_array_equal(t[i].double().cpu().numpy(), c)


def test_zero_fields_takes_odd_sizes_alignments_and_missing_components():
    desc, p, _ = _setup((3, 5, 7), (0, 0, 0), (0, 0, 0))
    n = int(np.prod(p.shape))
    for shift in (0, 1):
        store = torch.ones((2, n + 2), dtype=torch.float32, device="cuda")
        N.call("pic_zero_fields", desc, N.P3(store[0, shift:].data_ptr(), None, store[1, shift:].data_ptr()),
               N.stream_handle())
        assert int(store.sum()) == 2 * 2 and not bool(store[:, shift:shift + n].any())
