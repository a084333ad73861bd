"""The LBVH walk's evaluation at the edges of its slots of 16 particles: states
of one walk group (at most 64 particles) and of a few, whose forces are direct
sums because every cell holds the group (theta tiny), against FP64.

Tolerance: an entry's term is a product of an FP32 difference and 1/s^3 from
v_rsq_f32, wrong by at most 15 u (u = 2^-24) of its size; at most 64 are added
in plain FP32, whose rounding walks about sqrt(64) u.  1.4e-6 of the sum of
the terms' magnitudes; 2e-6 is allowed."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu
EPS = 1e-2


@pytest.mark.parametrize("acc_mode", [L.SF_ACC_REFERENCE, L.SF_ACC_PHYSICAL])
@pytest.mark.parametrize("quad", [0, 1])
@pytest.mark.parametrize("N", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 129, 300])
def test_slots_close_to_fp64(N, quad, acc_mode):
    print(f"walk slots N={N} quad={quad} acc_mode={acc_mode}", flush=True)
    rng = np.random.default_rng(N)
    with Simulation(N, enable_tree=1, tree_mode=L.SF_TREE_LBVH, theta=1e-6, leaf_size=3, quadrupole=quad, logging=0,
                    epsilon=EPS, precision=L.SF_PRECISION_FAST, acc_mode=acc_mode) as s:
        s.pos[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.mas[:] = rng.uniform(0.5, 1.5, N).astype(np.float32)
        s.solve()
        x, m = s.pos.astype(np.float64), s.mas.astype(np.float64)
        acc, pot = s.acc.astype(np.float64), s.pot.astype(np.float64)
    L.set_params()
    for i in range(N):
        d = x - x[i]
        s2 = (d * d).sum(1) + EPS * EPS
        w = m * s2 ** -1.5 * (m[i] if acc_mode == L.SF_ACC_REFERENCE else 1.0)
        assert np.abs(acc[i] - w @ d).max() <= 2e-6 * (w * np.sqrt((d * d).sum(1))).sum(), i
        p = (m / np.sqrt(s2)).sum()
        assert abs(pot[i] + p) <= 2e-6 * p, i


@pytest.mark.parametrize("N", [65535, 65536, 65537, 131072, 230001, 400000])
def test_every_group_is_walked(N):
    """The group list at the edges of its blocks (65536 positions) and with
    more groups than wavefronts.  A cell is accepted from d > l / theta + its
    centre's offset, so its monopole is wrong by at most 3 (theta / 2)^2 =
    0.12 of its size; a particle of a group left out would keep pot = 0."""
    print(f"walk groups N={N}", flush=True)
    rng = np.random.default_rng(N)
    with Simulation(N, enable_tree=1, tree_mode=L.SF_TREE_LBVH, theta=0.4, leaf_size=3, logging=0, epsilon=EPS,
                    precision=L.SF_PRECISION_FAST, acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.mas[:] = np.float32(1.0 / N)
        s.solve()
        x, m = s.pos.astype(np.float64), s.mas.astype(np.float64)
        acc, pot = s.acc.astype(np.float64), s.pot.astype(np.float64)
    L.set_params()
    assert pot.max() < 0.0
    for i in np.linspace(0, N - 1, 24).astype(int):
        d = x - x[i]
        s2 = (d * d).sum(1) + EPS * EPS
        w = m * s2 ** -1.5
        assert np.abs(acc[i] - w @ d).max() <= 0.12 * (w * np.sqrt((d * d).sum(1))).sum(), i
        p = (m / np.sqrt(s2)).sum()
        assert abs(pot[i] + p) <= 0.12 * p, i
