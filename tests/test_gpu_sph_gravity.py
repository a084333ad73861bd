"""sim_solv of the exact policy with the reference SPH model, whose gravity and
density share a launch up to 5120 particles, against the two solvers called one
after the other: the same bits, at the edges of the blocks of 32 particles and
of that range, for every choice of the compensated sums and of acc."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def run(N, acc_mode, kahan, apart):
    rng = np.random.default_rng(N)
    with Simulation(N, enable_tree=0, enable_sph=1, logging=0, epsilon=1e-2, acc_mode=acc_mode,
                    kahan_solver=kahan & 1, kahan_energy=kahan >> 1) as s:
        s.pos[:] = rng.normal(scale=0.6, size=(N, 3)).astype(np.float32)
        s.mas[:] = rng.uniform(0.5, 1.5, N).astype(np.float32) / N
        s.rad[:] = rng.uniform(0.05, 0.3, N).astype(np.float32)
        if apart:
            s.solve_gravity_pp()
            s.solve_sph()
        else:
            s.solve()
        out = [np.array(a, copy=True).view(np.uint32) for a in (s.acc, s.pot, s.rho, s.prs)]
    L.set_params()
    return out


@pytest.mark.parametrize("N,acc_mode,kahan",
                         [(N, L.SF_ACC_REFERENCE, 3) for N in (1, 31, 33, 64, 1000, 5120, 5121, 8193)]
                         + [(129, a, k) for a in (L.SF_ACC_REFERENCE, L.SF_ACC_PHYSICAL) for k in range(4)])
def test_shared_launch_has_the_same_bits(N, acc_mode, kahan):
    print(f"sph gravity N={N} acc_mode={acc_mode} kahan={kahan}", flush=True)
    for a, b in zip(run(N, acc_mode, kahan, False), run(N, acc_mode, kahan, True)):
        assert np.array_equal(a, b)
