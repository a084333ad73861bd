"""The partial sums of the kernels that split a body's sum over blocks, on
states whose terms are whole numbers: everything that is added in FP32 stays
below 2^24 and is exact; what a block hands to the combine may be odd and
larger, and is exact only if it is held in more than 24 bits.  The result is
then the rounded exact sum, bit for bit.

Bodies of even index are sources at (1, 0, 0), those of odd index massless
targets at the origin: s^2 rounds to 1 and a term is the source's mass, a
number of 18 bits.  The sources of every second set (of 256 or 1024 bodies)
lie at (-1, 0, 0) instead, so that the sums of the sets cancel.  Checked are
the targets at the middle of a tile, whose j sums take half of their terms
from each of the two copies."""
import numpy as np
import pytest
import torch

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -20


def sources(N, set_size):
    """index, sign and value of the sources, and the targets that are checked"""
    i = np.arange(N)
    src = i % 2 == 0
    sign = np.where((i // set_size) % 2 == 0, 1.0, -1.0)
    value = np.random.default_rng(N).integers(2 ** 17, 2 ** 18, N).astype(np.float64)
    rows = np.flatnonzero(~src & (abs(i % 64 - 31) <= 2))
    return src, sign, value, rows


@pytest.mark.parametrize("N,set_size", [(12200, 256), (26500, 1024), (67500, 1024), (300950, 1024)])
def test_force_of_whole_numbers_is_exact(N, set_size):
    print(f"whole-number force N={N}", flush=True)
    src, sign, value, rows = sources(N, set_size)
    with Simulation(N, enable_tree=0, logging=0, epsilon=EPS, precision=L.SF_PRECISION_FAST,
                    acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = 0
        s.pos[src, 0] = sign[src]
        s.mas[:] = np.where(src, value, 0.0)
        s.solve_gravity_pp()
        got = s.acc[rows].copy()
    L.set_params()
    want = np.float32((sign * value)[src].sum())
    assert abs(want) < 2 ** 25
    assert np.all(got[:, 0] == want), np.unique(got[:, 0] - want)
    assert np.all(got[:, 1:] == 0)


@pytest.mark.parametrize("masses", ["equal", "general"])
@pytest.mark.parametrize("N", [12200, 140200])
def test_vjp_of_whole_numbers_is_exact(N, masses):
    """The weights take the masses' place: nu_j along y, across the distance,
    so that a term of g is m_k nu_j - m_j nu_k = nu_j."""
    print(f"whole-number VJP N={N} masses={masses}", flush=True)
    src, sign, value, rows = sources(N, 256)
    pos, mu = np.zeros((2, N, 3), np.float32)
    pos[src, 0] = 1
    mu[src, 1] = (sign * value)[src]
    mas = np.ones(N, np.float32)
    if masses == "general":
        mas[src] = np.random.default_rng(N + 1).uniform(0.5, 1.5, N)[src].astype(np.float32)
    lib = L.load()
    L.set_params(epsilon=EPS, acc_mode=L.SF_ACC_PHYSICAL)
    x, m, u = (torch.from_numpy(a).cuda() for a in (pos, mas, mu))
    g = torch.empty_like(x)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.sf_force_vjp_dev(N, x.data_ptr(), m.data_ptr(), u.data_ptr(), g.data_ptr(), stream) == 0
    got = g.cpu().numpy()[rows]
    L.set_params()
    want = np.float32((sign * value)[src].sum())
    assert abs(want) < 2 ** 25
    assert np.all(got[:, 1] == want), np.unique(got[:, 1] - want)
    assert np.all(got[:, [0, 2]] == 0)


@pytest.mark.parametrize("seed", range(8))
def test_walk_of_whole_numbers_is_exact(seed):
    """The LBVH walk's sums over list entries: 40 targets at the origin, 256
    sources at distance 1 (to the last bit of s^2) that a tiny theta opens, so
    that a target's potential is the rounded sum of the sources' masses."""
    print(f"whole-number walk seed={seed}", flush=True)
    k = np.arange(256)
    value = np.random.default_rng(seed).integers(2 ** 16, 2 ** 17, 256) * 2 + 1
    with Simulation(296, logging=0, epsilon=EPS, theta=1e-9, precision=L.SF_PRECISION_FAST, tree_mode=L.SF_TREE_LBVH,
                    acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = 0
        s.pos[40:] = np.stack([np.ones(256), (k % 16) * 2.0 ** -20, (k // 16) * 2.0 ** -20], 1)
        s.mas[:40] = 0
        s.mas[40:] = value
        s.solve()
        got = s.pot[:40].copy()
    L.set_params()
    want = np.float32(-value.sum())
    assert np.all(got == want), np.unique(got - want)
