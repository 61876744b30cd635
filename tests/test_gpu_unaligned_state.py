"""A state that is not 16-byte aligned (a view into a larger array): integrate takes the steps of
hrw_rktvd_steps_noalloc, bit for bit, as it does on aligned ones."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER, ZG = 0, 1
LF, GOD = 0, 1


@pytest.mark.parametrize("arith", ["fast", "exact"])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [8, 300, 5000, 50021])
@pytest.mark.parametrize("flux,bc", [(LF, PER), (GOD, ZG)])
def test_integrate(hh, dev, arith, shift, n, flux, bc):
    import torch
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    u0 = torch.as_tensor(0.4 + np.sin(math.pi * x + 0.3) + 0.5 * (x > 0.2), device=dev)
    dt = 0.2 * (2.0 / n) / 2.5
    p = hh.Burgers1D(n, flux=flux, bc=bc, arith=arith)
    a, b = (torch.zeros(n + 4, dtype=torch.float64, device=dev)[shift:shift + n] for _ in range(2))
    assert a.data_ptr() % 16 == (shift % 2) * 8
    a.copy_(u0)
    b.copy_(u0)
    hh.RkTvd(p, order=3).integrate(a, 0.0, 39.5 * dt, dt)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    hh._lib.call("hrw_rktvd_steps_noalloc", p._h, 3, C.c_void_p(b.data_ptr()), 40, dt, stream)
    torch.cuda.synchronize()
    assert torch.equal(a, b)
