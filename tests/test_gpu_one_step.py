"""Calls of one step on a state advanced in place, over several blocks: a block must not store its
result before its neighbours have read its cells.  Against one launch per stage (a problem tuned to a
kernel, a batch with set_cells_per_lane), bit for bit."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER, ZG = 0, 1
LF, GOD = 0, 1


def u0(n, seed=5):
    rng = np.random.default_rng(seed + n)
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    return 0.4 + np.sin(math.pi * x + 0.3) + 0.5 * (x > 0.2) + 0.05 * rng.standard_normal(n)


def line(hh, dev, n, flux, bc, alpha, arith, order, tuned, calls, tape):
    import torch
    p = hh.Burgers1D(n, 3, 1e-6, flux=flux, bc=bc, alpha=alpha, arith=arith)
    if tuned:
        p.tune(0, 4)
    ode = hh.RkTvd(p, order=order)
    if tape:
        ode.tape(1)
    dt = 0.2 * (2.0 / n) / 2.5
    u = torch.as_tensor(u0(n), device=dev).clone()
    t = 0.0
    for _ in range(calls):
        t = ode.integrate(u, t, t + 0.5 * dt, dt)
    assert ode.fevals == calls * order
    return u.cpu().numpy()


@pytest.mark.parametrize("n", [622, 1117, 5000, 50021, 1000003])
@pytest.mark.parametrize("flux,bc,alpha", [(GOD, PER, -1.0), (GOD, ZG, -1.0), (LF, PER, 2.5), (LF, PER, -1.0)])
@pytest.mark.parametrize("arith", ["fast", "exact"])
@pytest.mark.parametrize("order", [2, 3])
def test_line(hh, dev, n, flux, bc, alpha, arith, order):
    a = line(hh, dev, n, flux, bc, alpha, arith, order, False, 4, False)
    assert np.array_equal(a, line(hh, dev, n, flux, bc, alpha, arith, order, True, 4, False))


@pytest.mark.parametrize("n", [1117, 50021])
@pytest.mark.parametrize("flux,bc,alpha", [(GOD, PER, -1.0), (GOD, ZG, -1.0), (LF, PER, 2.5)])
def test_recorded_line(hh, dev, n, flux, bc, alpha):
    a = line(hh, dev, n, flux, bc, alpha, "fast", 3, False, 4, True)
    assert np.array_equal(a, line(hh, dev, n, flux, bc, alpha, "fast", 3, True, 4, False))


@pytest.mark.parametrize("n", [5000, 50021])
@pytest.mark.parametrize("flux,bc", [(GOD, ZG), (LF, PER)])
@pytest.mark.parametrize("steps", [1, 3])
@pytest.mark.parametrize("shift", [0, 2, 640])
def test_adjoint_forward_in_place(hh, dev, n, flux, bc, steps, shift):
    """The result over the initial state, or over a part of it."""
    import torch
    dt = 0.2 * (2.0 / n) / 2.5
    adj = hh.Adjoint(hh.Burgers1D(n, flux=flux, bc=bc, alpha=2.5), nsteps=steps, dt=dt)
    buf = torch.zeros(n + shift, dtype=torch.float64, device=dev)
    buf[:n] = torch.as_tensor(u0(n), device=dev)
    g = torch.as_tensor(u0(n, 9), device=dev)
    ref = adj.forward(buf[:n]).clone()
    gref = adj.backward(g).clone()
    out = buf[shift:]
    adj.forward(buf[:n], out)
    assert torch.equal(out, ref) and torch.equal(adj.backward(g), gref)


@pytest.mark.parametrize("flux,alpha", [(GOD, -1.0), (LF, 2.5), (LF, -1.0)])
@pytest.mark.parametrize("steps,calls", [(1, 4), (65, 1)])
def test_batch(hh, dev, flux, alpha, steps, calls):
    """More blocks than the chip holds: the later blocks of a line start after earlier ones have ended."""
    import torch
    ns = [20000] * 240 + [61000] * 12 + [300, 40]
    us = [u0(n, i) for i, n in enumerate(ns)]
    dts = np.array([0.2 * (2.0 / n) / 2.5 for n in ns])
    res = []
    for fixed in (False, True):
        b = hh.BurgersBatch(ns, [2 + i % 2 for i in range(len(ns))], dts, flux=flux, alpha=alpha)
        if fixed:
            b.set_cells_per_lane(6)
        u = b.pack(us, dev)
        for _ in range(calls):
            b.step(u, steps)
        torch.cuda.synchronize()
        res.append((u.cpu().numpy(), b.t.copy()))
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])
