"""The PP step whose kicks and drift ride on the force's launches against the
one that makes them in launches of their own (the step times log needs them
apart): the same operations, so the same bits.  Sizes at the edges of the
blocks and of the two force kernels' ranges; a position that the host changes
between steps restarts its FP64 track in both."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def run(N, acc_mode, out_dir):
    rng = np.random.default_rng(N)
    kw = dict(logging=1, out_dir=str(out_dir)) if out_dir else dict(logging=0)
    with Simulation(N, enable_tree=0, precision=L.SF_PRECISION_FAST, acc_mode=acc_mode, dt=1e-2, **kw) as s:
        s.pos[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.vel[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.mas[:] = (rng.uniform(0.5, 1.5, N) / N).astype(np.float32)
        s.solve_gravity_pp()
        s.step()
        s.step()
        s.pos[N // 2] += np.float32(0.125)
        s.step()
        out = [np.array(a, copy=True) for a in (s.pos, s.vel, s.acc, s.pot, s.ken, s.pen)]
    L.set_params()
    return out


@pytest.mark.parametrize("acc_mode", [L.SF_ACC_REFERENCE, L.SF_ACC_PHYSICAL])
@pytest.mark.parametrize("N", [1, 63, 1025, 9216, 9217, 24577])
def test_fused_step_has_the_same_bits(N, acc_mode, tmp_path):
    print(f"fused step N={N} acc_mode={acc_mode}", flush=True)
    for a, b in zip(run(N, acc_mode, None), run(N, acc_mode, tmp_path)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
