"""Mirror mode's transfers (one kernel for the ranges up to 1.3 MB, the copy
engine above) against the resident mode with whole-state transfers: the same
bits in every block, and nothing written that the call does not write.  Ragged
counts leave words before and after the 16-byte boundaries; 25206 and 25207
bodies are the last step by kernel and the first by the copy engine (13 blocks
of 4 bytes)."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu

NAMES = ("pos", "vel", "acc", "mas", "pot", "ken", "pen")


def run(N, mode, sph, call):
    rng = np.random.default_rng(N)
    names = NAMES + (("rad", "rho", "prs") if sph else ())
    with Simulation(N, enable_tree=0, enable_sph=sph, precision=L.SF_PRECISION_FAST, dt=1e-3, logging=0,
                    mem_mode=mode) as s:
        for k in names:
            a = getattr(s, k)
            a[:] = rng.uniform(0.5, 1.5, a.shape).astype(np.float32)
        if mode == L.SF_MEM_RESIDENT:
            s.to_device()
        getattr(s, call)()
        st = s.stats() if call == "step" else None
        if mode == L.SF_MEM_RESIDENT:
            s.to_host()
        out = {k: np.array(getattr(s, k), copy=True).view(np.uint32) for k in names}
    L.set_params()
    return out, st


@pytest.mark.parametrize("call", ["solve", "step"])
@pytest.mark.parametrize("N,sph", [(1, 0), (2, 0), (3, 0), (5, 1), (1023, 0), (1026, 1), (25206, 0), (25207, 0)])
def test_mirror_equals_resident(N, sph, call):
    print(f"mirror N={N} sph={sph} {call}", flush=True)
    a, b = run(N, L.SF_MEM_MIRROR, sph, call), run(N, L.SF_MEM_RESIDENT, sph, call)
    for k in a[0]:
        assert np.array_equal(a[0][k], b[0][k]), k
    assert a[1] == b[1]
