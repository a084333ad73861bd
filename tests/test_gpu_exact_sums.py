"""The parallel forms of the reference's sequential FP64 Kahan sums
(device/exact_sum.hip), bit for bit against the sequence: the energies T and
V at the edges of a chunk of 4096 terms, over distributions that take the
integer sum and ones that do not (exponents spanning 27 and 28 binary
orders, non-finite terms), and the tree bounds' mean radius where the
interval around it leaves the float open."""
import numpy as np
import pytest

from starflood_amd import _lib as L
from starflood_amd.sim import Simulation

pytestmark = pytest.mark.gpu


def kahan(x):
    """src/simulation.c:455-497"""
    s = c = 0.0
    for v in x.astype(np.float64).tolist():
        y = v - c
        t = s + y
        c = (t - s) - y
        s = t
    return s


def terms(kind, N):
    rng = np.random.default_rng(N)
    x = rng.lognormal(sigma=2.0, size=N).astype(np.float32)
    if kind == "mixed":
        x *= rng.choice([-1, 1], N).astype(np.float32)
        x[::7] = 0
    elif kind in ("span27", "span28"):     # greatest and least exponents that far apart
        x = np.ldexp(1 + rng.random(N), rng.integers(0, 27, N)).astype(np.float32)
        x[0], x[-1] = np.float32(1.0 + 2.0 ** -23), np.ldexp(np.float32(1.75), int(kind[4:]))
    elif kind == "wide":
        x = (rng.choice([-1, 1], N) * np.ldexp(1 + rng.random(N), rng.integers(-60, 60, N))).astype(np.float32)
    elif kind == "subnormal":
        x = (rng.integers(1, 2 ** 23, N) * 2.0 ** -149).astype(np.float32)
    elif kind == "zero":
        x[:] = 0
        x[::2] = -0.0
    elif kind == "inf":
        x[N // 2] = np.inf
    return x


@pytest.mark.parametrize("kind", ["plain", "mixed", "span27", "span28", "wide", "subnormal", "zero", "inf"])
@pytest.mark.parametrize("N", [2, 255, 4095, 4096, 4097, 20000])
def test_energies_equal_the_sequence(kind, N):
    print(f"energy sums N={N} {kind}", flush=True)
    with Simulation(N, enable_tree=0, logging=0) as s:
        s.ken[:] = terms(kind, N)
        s.pen[:] = -terms("plain", N)[::-1]
        st = s.stats()
        want = kahan(s.ken), kahan(s.pen)
    for got, w in zip((st["T"], st["V"]), want):
        assert np.float64(got).tobytes() == np.float64(w).tobytes() or (np.isnan(got) and np.isnan(w))
    L.set_params()


def cube(a, jit):
    return np.stack([(-2.0 * a + 0.5 * j * a).astype(np.float32) for j in jit] +
                    [(2.0 * a + 0.5 * j * a).astype(np.float32) for j in jit])


def test_bounds_where_the_interval_leaves_the_float_open(oracle):
    """One particle: the mean is its radius times 1.0.  Radii whose interval
    of 16 u straddles a rounding boundary of a bound (about three of the 2^23
    in a binade, by the step's jitter) take the sequence."""
    r = 1.0 + np.arange(2 ** 23) * 2.0 ** -23
    d = 16.0 * 2.0 ** -53
    rows = [(0, 1.0), (0, 1.2345678)]
    for step in range(6):
        u4 = oracle.pcg4d([0x638FE17B + step, 0xB10BDCE7, 0x7B8ADB9B, 0xD8C5850E])
        jit = [2.0 * (2.3283062977608182109179324470460414886474609375e-10 * float(v)) - 1.0 for v in u4[:3]]
        hits = np.flatnonzero((cube(r * (1 - d), jit) != cube(r * (1 + d), jit)).any(0))
        rows += [(step, r[k]) for k in hits[:4]]
    print(f"mean radius: {len(rows) - 2} open radii", flush=True)
    assert len(rows) > 4
    for step, v in rows:
        with Simulation(1, logging=0) as s:
            s.pos[:] = [[v, 0, 0]]
            s.mas[:] = 1
            s.step_number = step
            s.solve()
            got = np.array(list(s.sim.tree.bounds), np.float32)
            want = np.zeros(6, np.float32)
            oracle.lib().orc_tree_bounds_ref(1, oracle.fp(s.pos.copy()), step, oracle.fp(want))
        assert np.array_equal(got, want), (step, v)
    L.set_params()


@pytest.mark.parametrize("N", [2, 511, 513, 300000])
def test_bounds_equal_the_oracle(oracle, N):
    print(f"mean radius N={N}", flush=True)
    pos = np.random.default_rng(N).normal(size=(N, 3)).astype(np.float32)
    with Simulation(N, logging=0, tree_nodes_max=1 << 19) as s:
        s.pos[:] = pos
        s.mas[:] = 1.0 / N
        s.step_number = 3
        s.solve()
        got = np.array(list(s.sim.tree.bounds), np.float32)
    want = np.zeros(6, np.float32)
    oracle.lib().orc_tree_bounds_ref(N, oracle.fp(pos), 3, oracle.fp(want))
    assert np.array_equal(got, want)
    L.set_params()
