"""The adjoint's forward phase forms each node value of J by itself, q w v times
the node's own weight, on 1-D and 2-D first-order grids too.

Isolated particles on a grid of spacing 1, zero fields: every product and sum
below is one FP32 rounding whichever way the compiler fuses it, so the node
values follow bit for bit from the stored position and the pushed velocity."""

import numpy as np
import pytest
import torch

from pypic3d_amd import workloads
from pypic3d_amd.adjoint import AdjointRun
from pypic3d_amd.particles.particle_class import SpeciesConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(64, 1, 1), (24, 32, 1)])
def test_node_values_are_products_of_their_own_weight(n):
    f = np.float32
    dims = 1 if n[1] == 1 else 2
    static, dyn = workloads.make_parameters(n, wind=tuple(float(m) for m in n), dt=0.25)
    rng = np.random.default_rng(7)
    cells = np.stack(np.meshgrid(*[np.arange(2, m - 2, 4) if m > 1 else np.array([0]) for m in n], indexing="ij"),
                     -1).reshape(-1, 3)
    P = len(cells)
    x = np.zeros((3, 1, P))
    for a in range(dims):
        x[a, 0] = cells[:, a] + rng.uniform(0.3, 0.7, P) - n[a] / 2
    x = x.astype(f)
    v = rng.uniform(-0.3, 0.3, (3, 1, P)).astype(f)
    cfg = SpeciesConfig(charge=np.array([-1.0]), mass=np.array([1.0]), weight=np.array([0.375]),
                        update_x=np.ones((1, 3), bool), update_u=np.ones((1, 3), bool))
    g = int(static.guard_cells)
    zero = torch.zeros((3,) + tuple(m + 2 * g for m in n), dtype=torch.float32, device="cuda")
    run = AdjointRun(static, dyn, cfg, torch.ones((1, P), dtype=torch.bool, device="cuda"))
    run.forward(torch.tensor(x, device="cuda"), torch.tensor(v, device="cuda"), zero, zero.clone(), 1)
    r = run.runner
    J = [c.cpu().numpy() for c in r.J]
    u = r.vel[r.cur][:, 0].cpu().numpy()                       # the pushed velocity of the step
    d = r.desc
    pre = f(0.375 / 0.25)                                      # -q w / (d_p d_q dt)
    q_dv = f(-0.375)
    lo, D, at = [], [], []
    for a in range(dims):
        i = np.floor((x[a, 0].astype(np.float64) - d.org_c[a]) / d.sp_c[a]).astype(int)
        lo.append((x[a, 0] - (i * d.sp_c[a] + d.org_c[a]).astype(f)).astype(f))
        D.append(u[a] * f(0.25))
        at.append(i)
        new = np.floor((x[a, 0].astype(np.float64) + u[a].astype(np.float64) * 0.25 - d.org_c[a]) / d.sp_c[a])
        assert (new == i).all()                                # nobody leaves its cell
    weight = [[(f(1) - lo[a]) - f(0.5) * D[a], lo[a] + f(0.5) * D[a]] for a in range(dims)]
    for side in range(2):
        if dims == 2:
            np.testing.assert_array_equal(J[0][at[0], at[1] + side, g], pre * -D[0] * weight[1][side])
            np.testing.assert_array_equal(J[1][at[0] + side, at[1], g], pre * -D[1] * weight[0][side])
        else:
            for c in (1, 2):
                np.testing.assert_array_equal(J[c][at[0] + side, g, g], q_dv * u[c] * weight[0][side])
