"""The step times log (timings_sim_step.csv): each phase's time in its own
column.  Sums and passes that take tens of microseconds show in ken_sum and
pen_sum, where two events in a row would show about two."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def times(tmp_path, N, mas, **kw):
    rng = np.random.default_rng(N)
    with Simulation(N, logging=1, out_dir=str(tmp_path), dt=1e-3, **kw) as s:
        s.pos[:] = rng.normal(size=(N, 3))
        s.vel[:] = rng.normal(size=(N, 3))
        s.mas[:] = mas
        if kw.get("mem_mode") == L.SF_MEM_RESIDENT:
            s.to_device()
        for _ in range(3):
            s.step()
    L.set_params()
    head, *rows = [r.split(",") for r in (tmp_path / "timings_sim_step.csv").read_text().splitlines()]
    return dict(zip(head, map(float, rows[-1])))


def test_exact_log_has_both_sums(tmp_path):
    """Terms whose exponents are too far apart for the integer sums: each sum is
    a sequence of 20000 steps of four dependent FP64 additions, over 100 us."""
    N = 20000
    print(f"exact step times N={N}", flush=True)
    mas = np.full(N, 1.0 / N, np.float32)
    mas[0] = 1e-20
    t = times(tmp_path, N, mas, enable_tree=0, precision=L.SF_PRECISION_EXACT)
    assert t["ken_sum"] > 100 and t["pen_sum"] > 100, t


def test_fast_log_has_the_sums_apart_from_the_kick(tmp_path):
    """The kick and the energy terms move 52 bytes a particle, the sums read 52:
    ken_sum is not a small part of kick_1."""
    N = 1 << 22
    print(f"fast step times N={N}", flush=True)
    t = times(tmp_path, N, 1.0 / N, enable_tree=1, tree_mode=L.SF_TREE_LBVH, precision=L.SF_PRECISION_FAST,
              acc_mode=L.SF_ACC_PHYSICAL, epsilon=1e-2, mem_mode=L.SF_MEM_RESIDENT)
    assert t["ken_sum"] > 0.25 * t["kick_1"], t
