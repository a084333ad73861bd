"""The radix sort through the LBVH build: the keys come out sorted and equal
keys in index order, at the edges of its tiles (1024 pairs up to 524288, 4096
above), with one digit value in whole tiles (clustered positions), many equal
keys, and more tiles than run at once."""
import ctypes as C

import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["normal", "clustered", "equal"])
@pytest.mark.parametrize("N", [1, 1023, 1025, 4095, 4097, 65537, 524288, 524289, 700001, 3000001])
def test_keys_sorted_and_stable(N, kind):
    print(f"radix N={N} kind={kind}", flush=True)
    rng = np.random.default_rng(N)
    with Simulation(N, enable_tree=1, tree_mode=L.SF_TREE_LBVH, theta=1.0, logging=0, epsilon=1e-2,
                    precision=L.SF_PRECISION_FAST) as s:
        x = rng.normal(size=(N, 3)).astype(np.float32)
        if kind == "clustered":
            x *= np.float32(1e-4)
            x[0] = 100.0
        elif kind == "equal":
            x = x[rng.integers(0, max(1, N // 1000), N)]
        s.pos[:] = x
        s.mas[:] = np.float32(1.0 / N)
        L.check(s.lib.tree_build(C.byref(s.sim.tree), N, s.pos.ctypes.data, s.mas.ctypes.data), "tree_build")
        tree = s.lbvh_export()
        keys, order = tree["keys"], tree["order"].astype(np.int64)
    L.set_params()
    assert np.array_equal(np.sort(order), np.arange(N))
    assert (keys[1:] >= keys[:-1]).all()
    assert (order[1:][keys[1:] == keys[:-1]] > order[:-1][keys[1:] == keys[:-1]]).all()
