"""A forked child reads and writes its own copy of sim.mem, as it does of any
other memory, though the runtime keeps page-locked memory out of children; the
parent's state is untouched and steps on.  1 particle lies inside a page;
161000 are just below the 8 MiB up to which the memory is copied."""
import os

import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 1000, 161000])
def test_forked_child_has_its_own_copy(N):
    print(f"fork N={N}", flush=True)
    rng = np.random.default_rng(N)
    with Simulation(N, enable_tree=0, logging=0, precision=L.SF_PRECISION_FAST) as s, \
            Simulation(7, enable_tree=0, logging=0) as other:
        s.pos[:] = rng.normal(size=(N, 3))
        s.mas[:] = 1.0 / N
        s.vel[:] = 1   # a single particle moves too
        other.vel[:] = 3
        s.step()
        want = s.mem.copy()
        pid = os.fork()
        if pid == 0:   # only memory is touched here
            code = 1
            try:
                same = np.array_equal(s.mem.view(np.uint32), want.view(np.uint32)) and np.all(other.vel == 3)
                s.mem[:] = -1
                code = 0 if same and np.all(s.mem == -1) else 2
            finally:
                os._exit(code)
        _, status = os.waitpid(pid, 0)
        assert status == 0
        assert np.array_equal(s.mem.view(np.uint32), want.view(np.uint32))
        s.step()
        assert np.isfinite(s.mem).all() and not np.array_equal(s.mem, want)
    L.set_params()
