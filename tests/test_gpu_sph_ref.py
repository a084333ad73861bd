"""The reference SPH model's sums (device/sph.hip on device/order_chain.h) at
the edges of their split (32 and 64 particles a block, tiles of 64 bodies,
runs of 8) and where the divisors leave the fast quotient's range, against
the oracle.  Tolerances as for the model itself (test_gpu_sph.py): the
device's expf and glibc's are faithfully rounded but differ, so rho within 4
ulp, P within 8, the force within 2e-5 of its size."""
import numpy as np
import pytest

from conftest import ulp_diff
from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,h", [(1, "plain"), (7, "plain"), (33, "plain"), (64, "plain"), (129, "plain"),
                                 (129, "tiny"), (129, "huge"), (1000, "mixed"), (8192, "plain"), (8200, "mixed")])
def test_reference_sums_at_the_edges(oracle, N, h):
    print(f"sph_ref N={N} {h}", flush=True)
    rng = np.random.default_rng(N)
    pos = rng.normal(scale=0.6, size=(N, 3)).astype(np.float32)
    mas = rng.uniform(0.5, 1.5, N).astype(np.float32) / N
    rad = rng.uniform(0.05, 0.3, N).astype(np.float32)
    if h == "tiny":     # pi^(3/2) h^5 below 2^-60
        rad[:] = 1e-5
    elif h == "huge":   # and above 2^60
        rad[:] = 3e4
    elif h == "mixed":
        rad[3], rad[N // 2] = 3e4, 2e4
    acc0 = rng.normal(size=(N, 3)).astype(np.float32)
    rho, prs, acc = oracle.sph_ref(pos, mas, rad, acc0)
    with Simulation(N, enable_tree=0, enable_sph=1, logging=0, epsilon=1e-2, dt=1e-3) as s:
        s.pos[:] = pos
        s.mas[:] = mas
        s.rad[:] = rad
        s.acc[:] = acc0
        s.solve_sph()
        assert ulp_diff(s.rho, rho).max() <= 4
        assert ulp_diff(s.prs, prs).max() <= 8
        d, f = s.acc - acc0, acc - acc0
        # acc0 + f is rounded: half an ulp of acc0's size on either side
        scale = np.maximum(np.linalg.norm(f, axis=1), 1e-3 * np.linalg.norm(f, axis=1).max())
        slack = 2.0 ** -23 * np.maximum(np.abs(acc0).max(1), np.abs(acc).max(1)) * 3
        assert (np.linalg.norm(d - f, axis=1) <= 2e-5 * scale + slack).all()
    L.set_params()
