"""Calls of more steps than one whole-integration launch takes (1024): they go on from launch to launch,
forward, recorded and in reverse, with the results of one launch per stage (a problem tuned to a kernel),
bit for bit; also where some of the launches wait in vain."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER, ZG = 0, 1
LF, GOD = 0, 1


def u0(n):
    rng = np.random.default_rng(n)
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    return 0.4 + np.sin(math.pi * x + 0.3) + 0.02 * rng.standard_normal(n)


def line(hh, dev, n, flux, bc, order, steps, tuned, arith="fast"):
    import torch
    p = hh.Burgers1D(n, 3, 1e-6, flux=flux, bc=bc, arith=arith)
    if tuned:
        p.tune(0, 4)
    ode = hh.RkTvd(p, order=order)
    dt = 1e-3 * (2.0 / n)
    u = torch.as_tensor(u0(n), device=dev).clone()
    t = ode.integrate(u, 0.0, (steps - 0.5) * dt, dt)
    t = ode.integrate(u, t, t + 2.5 * dt, dt)
    return u.cpu().numpy(), t, ode.fevals, ode.istate


@pytest.mark.parametrize("polls", [None, "40"])
@pytest.mark.parametrize("n,order", [(100, 3), (100, 1), (2000, 3), (2000, 2)])
@pytest.mark.parametrize("flux,bc", [(LF, PER), (GOD, ZG)])
@pytest.mark.parametrize("steps", [1024, 1025, 2050])
def test_integrate(hh, dev, monkeypatch, polls, n, order, flux, bc, steps):
    ref = line(hh, dev, n, flux, bc, order, steps, True)
    if polls:
        monkeypatch.setenv("HRW_RESIDENT_POLLS", polls)
    out = line(hh, dev, n, flux, bc, order, steps, False)
    assert np.array_equal(out[0], ref[0]) and out[1:] == ref[1:] and out[2] == order * (steps + 3)


def test_exact_equals_oracle(oracle, hh, dev):
    import torch
    n, steps = 700, 1500
    u = u0(n)
    dt = 1e-3 * (2.0 / n)
    d = torch.as_tensor(u, device=dev).clone()
    hh.RkTvd(hh.Burgers1D(n, arith="exact"), order=3).integrate(d, 0.0, (steps - 0.5) * dt, dt)
    ref, _, taken, _ = oracle.burgers_rk(u, np.diff(oracle.grid_linear(-1.0, 1.0, n)), tout=(steps - 0.5) * dt, dt=dt)
    assert taken == steps and np.array_equal(d.cpu().numpy(), ref)


@pytest.mark.parametrize("at", [3, 1500])
def test_nonfinite_is_reported(hh, dev, at):
    """A state that leaves the finite numbers in whichever launch of the call."""
    import torch
    n = 300
    u = u0(n)
    ode = hh.RkTvd(hh.Burgers1D(n), order=3)
    d = torch.as_tensor(u, device=dev).clone()
    dt = 1e-3 * (2.0 / n)
    ode.integrate(d, 0.0, (at - 0.5) * dt, dt)
    d[5] = float("inf")
    with pytest.raises(hh.HrwError, match="non-finite"):
        ode.integrate(d, 0.0, (3000 - at - 0.5) * dt, dt)


@pytest.mark.parametrize("polls", [None, "40"])
@pytest.mark.parametrize("n,order", [(100, 3), (100, 1), (2000, 3), (2000, 2)])
@pytest.mark.parametrize("flux,bc,alpha", [(LF, PER, -1.0), (LF, ZG, -1.0), (GOD, ZG, -1.0)])
@pytest.mark.parametrize("steps", [1025, 2050])
def test_gradient(hh, dev, monkeypatch, polls, n, order, flux, bc, alpha, steps):
    import torch
    res = []
    for tuned in (True, False):
        if polls and not tuned:
            monkeypatch.setenv("HRW_RESIDENT_POLLS", polls)
        p = hh.Burgers1D(n, 3, 1e-6, flux=flux, bc=bc, alpha=alpha)
        if tuned:
            p.tune(0, 4)
        a = hh.Adjoint(p, nsteps=steps, dt=1e-3 * (2.0 / n), order=order, ckpt_every=steps)
        u = torch.as_tensor(u0(n), device=dev).clone()
        g = torch.cos(3 * u)
        a.forward(u, u)
        first = a.backward(g)
        a.backward(g, g)
        res.append((u, first, g))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    assert torch.equal(res[0][1], res[0][2]) and torch.equal(res[1][1], res[1][2])
