"""The force and the force VJP of small states (device/pp.hip's k_pp_few,
device/adjoint.hip's k_vjp) at the edges of their tiles of 64 bodies, of the
padding to 1024 and of the sizes where a wavefront takes another tile, with
equal masses, one that differs and general ones, against FP64.  The force of
the caller's arrays and the one of packed bodies (a step of dt = 0) have the
same bits.

Tolerances: a force term is an FP32 difference times 1/s^3 from v_rsq_f32,
wrong by at most 15 u (u = 2^-24); a tile's 64 are added plainly, walking about
sqrt(64) u: 1.4e-6 of the sum of the terms' magnitudes, 2e-6 allowed.  A VJP
term has 1/s^5 (23 u), w's difference of two rounded products (2 u of the
products) and d . w (5 u): 38 u and sqrt(64) u, 2.8e-6, 4e-6 allowed."""
import numpy as np
import pytest
import torch

from starflood_amd import _lib as L
from starflood_amd import adjoint as A
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu
EPS = 1e-2
SIZES = [1, 2, 63, 64, 65, 1023, 1024, 1025, 3000, 5120, 5121, 7200, 9216]


def state(N, masses):
    rng = np.random.default_rng(N)
    pos = rng.normal(size=(N, 3)).astype(np.float32)
    mas = np.full(N, np.float32(1.0 / 3.0) / N, np.float32)
    if masses == "one_differs":
        mas[N // 2] *= 2
    elif masses == "general":
        mas *= rng.uniform(0.5, 1.5, N).astype(np.float32)
    return pos, mas, rng.normal(size=(N, 3)).astype(np.float32)


@pytest.mark.parametrize("masses", ["equal", "one_differs", "general"])
@pytest.mark.parametrize("N", SIZES)
def test_force_close_to_fp64(N, masses):
    print(f"pp few N={N} masses={masses}", flush=True)
    pos, mas, _ = state(N, masses)
    L.set_params(epsilon=EPS, precision=L.SF_PRECISION_FAST, acc_mode=L.SF_ACC_PHYSICAL)
    acc, pot = A.force(torch.tensor(pos, device="cuda"), torch.tensor(mas, device="cuda"))
    acc, pot = acc.cpu().numpy(), pot.cpu().numpy()
    with Simulation(N, enable_tree=0, logging=0, epsilon=EPS, dt=0.0, precision=L.SF_PRECISION_FAST,
                    acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = pos
        s.mas[:] = mas
        s.step()
        assert np.array_equal(s.acc.view(np.uint32), acc.view(np.uint32))
        assert np.array_equal(s.pot.view(np.uint32), pot.view(np.uint32))
    L.set_params()
    x, m = pos.astype(np.float64), mas.astype(np.float64)
    for i in np.unique(np.r_[0, N // 2, N - 1, np.linspace(0, N - 1, 40).astype(int)]):
        d = x - x[i]
        s2 = (d * d).sum(1) + EPS * EPS
        w = m * s2 ** -1.5
        assert np.abs(acc[i] - w @ d).max() <= 2e-6 * (w * np.sqrt((d * d).sum(1))).sum(), i
        p = (m / np.sqrt(s2)).sum()
        assert abs(pot[i] + p) <= 2e-6 * p, i


@pytest.mark.parametrize("masses", ["equal", "one_differs", "general"])
@pytest.mark.parametrize("N", SIZES)
def test_vjp_close_to_fp64(N, masses):
    print(f"vjp few N={N} masses={masses}", flush=True)
    pos, mas, mu = state(N, masses)
    L.set_params(epsilon=EPS, precision=L.SF_PRECISION_FAST, acc_mode=L.SF_ACC_PHYSICAL)
    g = A.force_vjp(*(torch.tensor(a, device="cuda") for a in (pos, mas, mu))).cpu().numpy()
    L.set_params()
    x, m, n = pos.astype(np.float64), mas.astype(np.float64), mu.astype(np.float64)
    for k in np.unique(np.r_[0, N // 2, N - 1, np.linspace(0, N - 1, 40).astype(int)]):
        d = x[k] - x
        s2 = (d * d).sum(1) + EPS * EPS
        w = m[k] * n - m[:, None] * n[k]
        size = m[k] * np.abs(n).sum(1) + m * np.abs(n[k]).sum()   # of the two products
        ref = (w / s2[:, None] ** 1.5 - 3.0 * (d * w).sum(1)[:, None] * d / s2[:, None] ** 2.5).sum(0)
        bound = (size * (s2 ** -1.5 + 3.0 * (d * d).sum(1) * s2 ** -2.5))[np.arange(N) != k].sum()
        assert np.abs(g[k] - ref).max() <= 4e-6 * bound, k
