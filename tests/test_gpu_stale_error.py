"""An error that an earlier, unrelated runtime call left on the thread says nothing about the launches
of a later call: whole-integration launches that went through must not be taken for refused ones (the
call would go on a second time from what they wrote)."""
import ctypes as C
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LF, GOD = 0, 1


@pytest.fixture
def stale(dev):
    """leave() leaves an error on this thread (of a device number there is none of), clear() takes it
    away (torch would report it)."""
    import torch
    torch.cuda.synchronize()
    hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line))

    class Stale:
        def leave(self):
            assert hip.hipSetDevice(1 << 20) != 0 and hip.hipPeekAtLastError() != 0

        def clear(self):
            hip.hipGetLastError()
    yield Stale()
    hip.hipGetLastError()


def u0(n):
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    return 0.4 + np.sin(math.pi * x + 0.3) + 0.5 * (x > 0.2)


@pytest.mark.parametrize("n", [300, 5000])
@pytest.mark.parametrize("flux", [LF, GOD])
def test_integrate(hh, dev, stale, n, flux):
    import torch
    dt = 0.2 * (2.0 / n) / 2.5
    p = hh.Burgers1D(n, flux=flux)
    out = []
    for with_error in (False, True):
        ode = hh.RkTvd(p, order=3)
        u = torch.as_tensor(u0(n), device=dev).clone()
        torch.cuda.synchronize()
        for i in range(3):
            if with_error:
                stale.leave()
            ode.integrate(u, 4 * i * dt, (4 * i + 3.5) * dt, dt)
        out.append((u, ode.fevals))
    stale.clear()
    assert torch.equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("n", [300, 5000])
def test_adjoint_in_place(hh, dev, stale, n):
    import torch
    adj = hh.Adjoint(hh.Burgers1D(n), nsteps=4, dt=0.2 * (2.0 / n) / 2.5)
    u = torch.as_tensor(u0(n), device=dev)
    g = torch.cos(u)
    uN = torch.empty_like(u)
    refN = adj.forward(u).clone()
    ref = adj.backward(g).clone()
    torch.cuda.synchronize()
    stale.leave()
    adj.forward(u, uN)
    adj.backward(g, g)
    stale.clear()
    assert torch.equal(uN, refN) and torch.equal(g, ref)


def test_batch(hh, dev, stale):
    import torch
    ns = [300, 5000, 20000]
    dts = np.array([0.2 * (2.0 / n) / 2.5 for n in ns])
    out = []
    for with_error in (False, True):
        b = hh.BurgersBatch(ns, [3, 2, 3], dts)
        u = b.pack([u0(n) for n in ns], dev)
        torch.cuda.synchronize()
        for _ in range(3):
            if with_error:
                stale.leave()
            b.step(u, 3)
        out.append(u)
    stale.clear()
    assert torch.equal(out[0], out[1])
