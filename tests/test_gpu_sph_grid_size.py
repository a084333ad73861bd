"""The cell size of the SPH grid search comes from the largest smoothing length,
found over up to 256 blocks: one particle, at the first and last places of a
block and of the array, is ten times as wide as the others, so a search that
missed it would lose most of its partners.  Density of the grid search against
every pair, which add the same terms in another order: N FP32 terms in partial
sums of at most 128, 2e-5 relative (the model's bound against FP64)."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def density(N, wide, search):
    rng = np.random.default_rng(N)
    h = 1.2 * N ** (-1 / 3)
    with Simulation(N, enable_tree=0, enable_sph=1, sph_model=L.SF_SPH_CUBIC_IDEAL, sph_search=search, logging=0,
                    precision=L.SF_PRECISION_FAST) as s:
        s.pos[:] = rng.uniform(size=(N, 3)).astype(np.float32)
        s.mas[:] = np.float32(1.0 / N)
        s.rad[:] = np.float32(h)
        s.rad[wide] = np.float32(min(10 * h, 0.5))
        s.solve_sph()
        s.solve_sph()
        out = np.array(s.rho, copy=True)
    L.set_params()
    return out


@pytest.mark.parametrize("N,wide", [(1, 0), (256, 255), (257, 256), (5000, 0), (5000, 4863), (65537, 65536),
                                    (70001, 65535), (70001, 70000)])
def test_the_widest_particle_sets_the_cells(N, wide):
    print(f"sph grid N={N} wide={wide}", flush=True)
    a, b = density(N, wide, L.SF_SPH_SEARCH_GRID), density(N, wide, L.SF_SPH_SEARCH_ALL)
    assert (np.abs(a - b) <= 2e-5 * np.abs(b)).all()
