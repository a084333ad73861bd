"""The kernels that evaluate each pair once (device/pp_sym.hip), at the sizes
where their split can go wrong: the first size they take, ragged ends, the
last narrow and first wide layout, an odd and an even number of sets, and
states whose planes need two launches; with equal masses, one that differs
(in a tile of the middle) and general ones.

Tolerance: a term of the sum is a product of an FP32 difference and 1/s^3
from v_rsq_f32, wrong by at most 15 u (u = 2^-24); its plain partial sums
hold at most 128 terms, whose rounding walks about sqrt(128) u.  Together
1.6e-6 of the sum of the terms' magnitudes; 2e-6 is allowed."""
import numpy as np
import pytest
import torch

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu
EPS = 1e-2


def state(N, masses):
    rng = np.random.default_rng(N)
    pos = rng.normal(size=(N, 3)).astype(np.float32)
    mas = np.full(N, np.float32(1.0 / 3.0) / N, np.float32)
    if masses == "one_differs":
        mas[N // 2] *= 2
    elif masses == "general":
        mas *= rng.uniform(0.5, 1.5, N).astype(np.float32)
    return pos, mas


def check(pos, mas, acc, pot, rows):
    x, m = pos.astype(np.float64), mas.astype(np.float64)
    for i in rows:
        d = x - x[i]
        s2 = (d * d).sum(1) + EPS * EPS
        w = m * s2 ** -1.5
        size = (w * np.sqrt((d * d).sum(1))).sum()
        assert np.abs(acc[i] - w @ d).max() <= 2e-6 * size, i
        p = (m / np.sqrt(s2)).sum()
        assert abs(pot[i] + p) <= 2e-6 * p, i


@pytest.mark.parametrize("masses", ["equal", "one_differs", "general"])
@pytest.mark.parametrize("N", [9217, 10240, 12289, 24576, 24577, 26000])
def test_pairs_once_close_to_fp64(N, masses):
    print(f"pp_sym N={N} masses={masses}", flush=True)
    pos, mas = state(N, masses)
    with Simulation(N, enable_tree=0, logging=0, epsilon=EPS, precision=L.SF_PRECISION_FAST,
                    acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = pos
        s.mas[:] = mas
        s.solve_gravity_pp()
        rows = np.unique(np.r_[0, 255, 256, 1023, 1024, N // 2, N - 1, np.linspace(0, N - 1, 57).astype(int)])
        check(pos, mas, s.acc.astype(np.float64), s.pot.astype(np.float64), rows)
        first = s.acc.copy(), s.pot.copy()
        s.solve_gravity_pp()
        assert np.array_equal(first[0], s.acc) and np.array_equal(first[1], s.pot)
    L.set_params()


@pytest.mark.parametrize("N", [299008, 299999])
def test_pairs_once_in_two_launches(N):
    print(f"pp_sym N={N}", flush=True)
    pos, mas = state(N, "general")
    with Simulation(N, enable_tree=0, logging=0, epsilon=EPS, precision=L.SF_PRECISION_FAST,
                    acc_mode=L.SF_ACC_PHYSICAL) as s:
        s.pos[:] = pos
        s.mas[:] = mas
        s.solve_gravity_pp()
        check(pos, mas, s.acc.astype(np.float64), s.pot.astype(np.float64),
              np.linspace(0, N - 1, 25).astype(int))
    L.set_params()


@pytest.mark.parametrize("N", [10007, 26000])
def test_force_without_potential_has_the_same_acc(N):
    print(f"pp_sym without pot N={N}", flush=True)
    lib = L.load()
    L.set_params(epsilon=EPS, acc_mode=L.SF_ACC_PHYSICAL)
    x, m = (torch.from_numpy(a).cuda() for a in state(N, "one_differs"))
    out = [torch.full((N, 3), float("nan"), device="cuda") for _ in range(2)]
    pot = torch.empty(N, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for acc, p in zip(out, (pot.data_ptr(), None)):
        assert lib.sf_force_dev(N, x.data_ptr(), m.data_ptr(), acc.data_ptr(), p, stream) == 0
    assert torch.equal(out[0], out[1])
    L.set_params()


def vjp_rows(x, m, mu, rows):
    """FP64 g_k and, per k, the size of its terms."""
    for k in rows:
        d = x[k] - x
        s2 = (d * d).sum(1) + EPS * EPS
        w = m[k] * mu - m[:, None] * mu[k]
        size = m[k] * np.linalg.norm(mu, axis=1) + m * np.linalg.norm(mu[k])
        g = (w * s2[:, None] ** -1.5 - 3.0 * d * ((d * w).sum(1) * s2 ** -2.5)[:, None]).sum(0)
        yield k, g, (size * (s2 ** -1.5 + 3.0 * (d * d).sum(1) * s2 ** -2.5)).sum()


@pytest.mark.parametrize("N,masses", [(9217, "equal"), (10240, "general"), (12289, "one_differs"), (26000, "equal"),
                                      (140001, "general")])
def test_vjp_pairs_once_close_to_fp64(N, masses):
    """k_vjp_sym, over the same edges (140001 needs two launches): a term is a
    product of six rounded factors, 20 u, and the walk of 64-term sums adds
    less; 2e-6 of the terms' sizes is allowed."""
    print(f"vjp_sym N={N} masses={masses}", flush=True)
    lib = L.load()
    L.set_params(epsilon=EPS, acc_mode=L.SF_ACC_PHYSICAL)
    pos, mas = state(N, masses)
    mu = np.random.default_rng(N + 1).normal(size=(N, 3)).astype(np.float32)
    x, m, u = (torch.from_numpy(a).cuda() for a in (pos, mas, mu))
    g = torch.empty_like(x)
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.sf_force_vjp_dev(N, x.data_ptr(), m.data_ptr(), u.data_ptr(), g.data_ptr(), stream) == 0
    got = g.cpu().numpy().astype(np.float64)
    rows = np.unique(np.r_[0, 255, 256, N // 2, N - 1, np.linspace(0, N - 1, 27).astype(int)])
    for k, want, size in vjp_rows(pos.astype(np.float64), mas.astype(np.float64), mu.astype(np.float64), rows):
        assert np.abs(got[k] - want).max() <= 2e-6 * size, k
    L.set_params()
