"""The level-synchronous build of the reference octree at the edges of its
tiles (1024 particles, 256 slots), with particles outside the bounds, a node
of every particle but one, and uneven depths: node arrays, forces and
potentials bit-identical to the oracle's serial insertion and walk."""
import numpy as np
import pytest

from conftest import bits
from starflood_amd import _lib as L
from starflood_amd.sim import Simulation
from test_gpu_tree_ref import direct_build, plummer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [7, 10, 256, 1023, 1024, 1025, 2049, 20000])
def test_build_with_bodies_outside_matches_oracle(oracle, N):
    print(f"tree levels N={N}", flush=True)
    pos, mas = plummer(N, N)
    bounds = np.array([-0.7, -0.9, -1.1, 0.8, 0.75, 1.0], np.float32)   # not a cube, a third of the bodies outside
    rc, nn, raw = direct_build(pos, mas, bounds)
    orc, _, _, onn, oraw = oracle.tree_ref(pos, mas, 0, bounds=bounds)
    assert rc == 0 and orc == 0
    assert nn == onn and np.array_equal(raw, oraw)


@pytest.mark.parametrize("N,spread", [(1025, 1.0), (3000, 1e-3), (70001, 1.0)])
def test_solve_matches_oracle(oracle, N, spread):
    print(f"tree solve N={N} spread={spread}", flush=True)
    pos, mas = plummer(N, N)
    pos *= np.float32(spread)
    pos[N // 2] = (2.0, -1.5, 1.0)   # with a small spread: every other body in a few cells
    with Simulation(N, enable_tree=1, logging=0, epsilon=1e-2, dt=1e-3) as s:
        s.pos[:] = pos
        s.mas[:] = mas
        s.step_number = 3
        s.solve()
        rc, bounds, nodes, nn, raw = oracle.tree_ref(pos, mas, 3)
        assert rc == 0 and s.sim.tree.num_nodes == nn
        assert np.array_equal(s.tree_nodes(), raw)
        acc, pot = oracle.tree_walk_ref(pos, mas, nodes, 262144, 1e-2)
        assert np.array_equal(bits(s.acc.ravel()), bits(acc.ravel()))
        assert np.array_equal(bits(s.pot), bits(pot))
    L.set_params()
