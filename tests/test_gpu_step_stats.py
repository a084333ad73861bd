"""The sums that a step's own passes leave on the host (kick, energy terms and
reduction in one launch, the exact sums and the fold in the next, the copy
with the state's) against sf_get_stats, which makes them with other launches:
the same bits.  Sizes on both sides of a chunk of the exact sums (4096), with
fewer and with all 512 blocks of the reduction (from 131072), and every route
of sim_step; then what verbose prints."""
import ctypes as C

import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu
ROUTES = {"exact": dict(enable_tree=0, precision=L.SF_PRECISION_EXACT),
          "fast": dict(enable_tree=0, precision=L.SF_PRECISION_FAST),
          "fast_tree": dict(enable_tree=1, tree_mode=L.SF_TREE_LBVH, precision=L.SF_PRECISION_FAST)}


def state(s, N):
    rng = np.random.default_rng(N)
    s.pos[:] = rng.normal(size=(N, 3))
    s.vel[:] = rng.normal(size=(N, 3))
    s.mas[:] = rng.uniform(0.5, 1.5, N) / N


@pytest.mark.parametrize("route", ROUTES)
@pytest.mark.parametrize("N", [1, 257, 4096, 4097, 131073])
def test_step_leaves_the_sums_of_its_state(N, route):
    print(f"step stats N={N} {route}", flush=True)
    with Simulation(N, logging=0, dt=1e-2, **ROUTES[route]) as s:
        state(s, N)
        s.step()
        s.step()
        got, want = s.step_stats(), s.stats()
    L.set_params()
    for k in want:
        assert np.array_equal(np.float64(got[k]).view(np.uint64), np.float64(want[k]).view(np.uint64)), k


def test_no_statistics_without_a_copy_to_the_host():
    with Simulation(100, logging=0, mem_mode=L.SF_MEM_RESIDENT, **ROUTES["fast"]) as s:
        state(s, 100)
        s.to_device()
        for _ in range(2):
            with pytest.raises(RuntimeError):
                s.step_stats()
            s.step()
    L.set_params()


@pytest.mark.parametrize("N", [1000, 4097])
def test_verbose_prints_the_energies(N, capfd):
    with Simulation(N, logging=0, verbose=1, dt=1e-2, **ROUTES["exact"]) as s:
        state(s, N)
        s.step()
        C.CDLL(None).fflush(None)
        lines = dict(l.split(" = ") for l in capfd.readouterr().out.splitlines() if " = " in l)
        want = s.stats()
    L.set_params()
    for name, k in (("E (tot)", "E"), ("V (pot)", "V"), ("T (kin)", "T")):
        assert lines[name] == "% .15f" % want[k]
