"""The splat's wavefront per particle at particle counts that leave blocks
partly filled and frames smaller than its window: the particles lie at
distance 1 from the origin, so the camera does not depend on their number and
each one more adds its own samples, a nonnegative count of at most 128, to the
frame, whatever the others do."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation
from starflood_amd.vis import Visualization

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(1, 1), (5, 40), (17, 3), (16, 16), (64, 48)])
def test_particles_add_their_own_samples(size):
    print(f"vis splat {size}", flush=True)
    axes = np.concatenate([np.eye(3), -np.eye(3)]).astype(np.float32)
    last = np.zeros((size[1], size[0], 4), np.int64)
    for N in range(1, 10):
        with Simulation(N, enable_tree=0, logging=0, epsilon=1e-2, dt=1e-3) as s:
            s.pos[:] = axes[np.arange(N) % 6]
            s.pot[:] = -np.arange(1, N + 1, dtype=np.float32)
            s.to_device()
            s.step_number = 7
            with Visualization(*size) as v:
                v.draw(s)
                a = v.atomic.astype(np.int64).reshape(last.shape)
        L.set_params()
        own = a - last
        assert own.min() >= 0 and own[..., 3].sum() <= 128
        # a particle's samples share one colour
        n = own[..., 3]
        if n.sum():
            y, x = np.unravel_index(n.argmax(), n.shape)
            assert (own[..., :3] * n[y, x] == own[y, x, :3] * n[..., None]).all()
        last = a
    if size == (64, 48):
        assert last[..., 3].sum() == 9 * 128
