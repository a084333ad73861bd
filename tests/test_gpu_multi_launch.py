"""Forces and VJPs of several launches (planes beyond 512 MiB: the force from
186368 bodies, its VJP from 107520) whose combine ends the step or the adjoint's
recursion: only the last launch's may, with the sums of all of them.

The step: the same bits as with the kicks in launches of their own.  The
adjoint of one step: against force and VJP calls put together here.  Each
value is then a sum of three FP32 roundings (2^-24 each) of terms no larger
than the largest value, and x_1 may differ by one rounding, which changes K by
less than 3 |d| 2^-24 / s; 16 x 2^-24 of the largest value is allowed."""
import numpy as np
import pytest
import torch

from starflood_amd import _lib as L
from starflood_amd import adjoint as A
from test_gpu_step_fused import run

pytestmark = pytest.mark.gpu


def test_step_of_two_force_launches(tmp_path):
    N = 190001
    print(f"step in two launches N={N}", flush=True)
    for a, b in zip(run(N, L.SF_ACC_REFERENCE, None), run(N, L.SF_ACC_REFERENCE, tmp_path)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def close(a, b):
    a, b = a.double(), b.double()
    assert (a - b).abs().max() <= 16 * 2.0 ** -24 * b.abs().max()


@pytest.mark.parametrize("N", [110001, 190001])
def test_adjoint_of_several_launches(N):
    print(f"adjoint in several launches N={N}", flush=True)
    dt, h = 1e-2, np.float32(0.5) * np.float32(1e-2)
    L.set_params(epsilon=0.5, dt=dt, acc_mode=L.SF_ACC_PHYSICAL)
    g = torch.Generator().manual_seed(N)
    x0, v0, gx, gv = (torch.randn(N, 3, generator=g).cuda() for _ in range(4))
    m = (torch.rand(N, generator=g) / N + 0.5 / N).cuda()
    x, v = x0.clone().requires_grad_(), v0.clone().requires_grad_()
    x1, v1 = A.kdk(x, v, m, 1)
    torch.autograd.backward([x1, v1], [gx, gv])

    hf, dtf = float(h), float(np.float32(dt))
    vh = (v0.double() + hf * A.force(x0, m)[0].double()).float()
    w1 = (x0.double() + dt * vh.double()).float()
    close(x1.detach(), w1)
    close(v1.detach(), vh.double() + hf * A.force(w1, m)[0].double())
    lx = gx + A.force_vjp(w1, m, hf * gv)
    lv = (gv.double() + dtf * lx.double()).float()
    close(x.grad, lx + A.force_vjp(x0, m, hf * lv))
    close(v.grad, lv)
    L.set_params()
