"""The exact policy's step with its kicks in the drift's and the reduction's
passes against the one with a launch for each (the step times log needs them
apart): the same roundings, so the same bits, at the edges of the blocks and
of the exact sums' chunks."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def run(N, tree, out_dir):
    rng = np.random.default_rng(N)
    kw = dict(logging=1, out_dir=str(out_dir)) if out_dir else dict(logging=0)
    with Simulation(N, enable_tree=tree, precision=L.SF_PRECISION_EXACT, dt=1e-2, **kw) as s:
        s.pos[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.vel[:] = rng.normal(size=(N, 3)).astype(np.float32)
        s.mas[:] = (rng.uniform(0.5, 1.5, N) / N).astype(np.float32)
        s.step()
        s.step()
        st = s.stats()
        out = [np.array(a, copy=True).view(np.uint32) for a in (s.pos, s.vel, s.acc, s.pot, s.ken, s.pen)]
        sums = [st[k] for k in ("T", "V", "W", "P", "L", "K")]
    L.set_params()
    return out, sums


@pytest.mark.parametrize("tree", [0, 1])
@pytest.mark.parametrize("N", [1, 63, 257, 1000, 4097])
def test_passes_of_the_exact_step(N, tree, tmp_path):
    print(f"exact step N={N} tree={tree}", flush=True)
    a, b = run(N, tree, None), run(N, tree, tmp_path)
    for x, y in zip(a[0], b[0]):
        assert np.array_equal(x, y)
    for x, y in zip(a[1], b[1]):
        assert np.array_equal(np.asarray(x), np.asarray(y))
