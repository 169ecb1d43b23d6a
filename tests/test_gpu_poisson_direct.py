"""Direct passes of the Poisson solve (FP64 transforms) against the oracle's CG
and the kernel's own CG, over neighbour modes, reduced axes and sizes around the
16- and 32-wide tiles of the transforms."""

import numpy as np
import pytest
import torch

from oracle import pic_oracle as O
from pypic3d_amd import workloads
from pypic3d_amd.solvers.electrostatic_yee import last_solve_info, solve_poisson_with_conjugate_gradient
from tests.gpu_helpers import gpu_field, host, oracle_params, rel_err

pytestmark = pytest.mark.gpu
A = (slice(2, -2),) * 3


def _problem(n, bc, seed):
    static, dyn = workloads.make_parameters(n, wind=tuple(0.5 * (1 + 0.3 * a) * m for a, m in enumerate(n)), dt=0.05,
                                            electrostatic=True, current_deposition="direct", bc=bc)
    p = oracle_params(static, dyn)
    rng = np.random.default_rng(seed)
    cells = int(np.prod(n))
    half = rng.standard_normal(cells // 2).astype(np.float32).astype(np.float64)
    v = np.zeros(cells)
    v[:2 * (cells // 2)] = np.concatenate([half, -half])          # zero total: consistent where it must be
    rho = np.zeros(p.shape)
    rho[A] = rng.permutation(v).reshape(n)
    return static, dyn, p, rho


@pytest.mark.parametrize("n,bc", [
    ((33, 17, 20), (0, 0, 0)), ((16, 31, 32), (0, 0, 0)), ((64, 2, 3), (0, 0, 0)),
    ((15, 65, 6), (1, 0, 0)), ((14, 10, 33), (1, 1, 0)), ((20, 18, 17), (1, 1, 1)), ((9, 16, 24), (0, 1, 1)),
    ((130, 1, 1), (0, 0, 0)), ((1, 1, 47), (0, 0, 0)), ((48, 33, 1), (1, 0, 0)), ((1, 24, 16), (0, 0, 1)),
])
def test_direct_passes_match_the_oracle_and_cg(n, bc):
    """FP32 output of an FP64-accurate potential: 1e-6 of its scale, up to the
    constant of a singular operator."""
    static, dyn, p, rho = _problem(n, bc, sum(n))
    zero = np.zeros(p.shape)
    got = host(solve_poisson_with_conjugate_gradient(gpu_field(rho), gpu_field(zero), static, dyn))[A]
    passes, res = last_solve_info["iterations"], last_solve_info["residual_norm"]
    assert 1 <= passes <= 3
    assert res <= 1e-12 * max(np.linalg.norm(rho[A]), 1.0)
    want = O.solve_poisson_cg(rho, zero, p, tol=1e-12, max_iter=20000)[A]
    singular = sum(bc) <= 1
    mean = (lambda f: f - f.mean()) if singular else (lambda f: f)
    assert rel_err(mean(got), mean(want)) <= 1e-6


def test_small_iteration_limits_keep_the_unconverged_cg():
    static, dyn, p, rho = _problem((24, 20, 16), (0, 0, 0), 3)
    zero = np.zeros(p.shape)
    got = host(solve_poisson_with_conjugate_gradient(gpu_field(rho), gpu_field(zero), static, dyn, max_iter=12))[A]
    assert last_solve_info["iterations"] == 12
    want = O.solve_poisson_cg(rho, zero, p, tol=1e-13, max_iter=12)[A]
    # FP32 vectors of the inner solve against the oracle's FP64 ones after twelve iterations
    assert rel_err(got - got.mean(), want - want.mean()) <= 1e-4


def test_direct_passes_start_from_the_given_potential_and_keep_its_mean():
    static, dyn, p, rho = _problem((16, 18, 20), (0, 0, 0), 5)
    phi0 = np.zeros(p.shape)
    phi0[A] = 3.0 + np.random.default_rng(1).standard_normal((16, 18, 20))
    got = host(solve_poisson_with_conjugate_gradient(gpu_field(rho), gpu_field(phi0), static, dyn))[A]
    base = host(solve_poisson_with_conjugate_gradient(gpu_field(rho), gpu_field(np.zeros(p.shape)), static, dyn))[A]
    scale = np.abs(base).max() + 3.0
    assert abs(got.mean() - phi0[A].astype(np.float32).mean()) <= 1e-6 * scale
    assert np.abs((got - got.mean()) - (base - base.mean())).max() <= 1e-6 * scale
    bad = rho.copy()
    bad[A][0, 0, 0] = np.nan           # no pass is made on a residual that is not a number
    out = solve_poisson_with_conjugate_gradient(gpu_field(bad), gpu_field(phi0), static, dyn)
    assert torch.isfinite(out).all() and last_solve_info["iterations"] == 0
