"""The recording forward (one launch, the stage inputs and alphas written as it goes) and the
reverse of a run whose every stage input is kept, against one launch per stage -- a problem tuned
to a kernel (tune(0, 4)) takes those -- bit for bit, at the edges of their splits."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER, ZG = 0, 1
LF, GOD = 0, 1


def case(n, seed=11, peaks=1):
    rng = np.random.default_rng(seed + n)
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    u = 0.4 + np.sin(math.pi * x + 0.3) + 0.3 * np.sin(3 * math.pi * x) + 0.5 * (x > 0.2) + 1e-3 * rng.standard_normal(n)
    return u, np.cos(3 * x) + 0.1 * rng.standard_normal(n), 0.2 * (2.0 / n) / 2.5


def grad(hh, dev, n, k, flux, bc, order, steps, tuned, alpha=-1.0, arith="fast", u=None, reps=1):
    import torch
    p = hh.Burgers1D(n, k, 1e-6, flux=flux, bc=bc, alpha=alpha, arith=arith)
    if tuned:
        p.tune(0, 4)
    u0, g, dt = case(n)
    u0 = u0 if u is None else u
    a = hh.Adjoint(p, nsteps=steps, dt=dt, order=order)
    ud, gd = torch.as_tensor(u0, device=dev), torch.as_tensor(g, device=dev)
    for _ in range(reps):
        uN = a.forward(ud)
        g0 = a.backward(gd)
    assert np.array_equal(gd.cpu().numpy(), g)
    return uN.cpu().numpy(), g0.cpu().numpy()


def same(a, b):
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), np.abs(a[1] - b[1]).max()


FORMS = [(LF, PER, -1.0), (LF, PER, 2.5), (LF, ZG, -1.0), (LF, ZG, 2.5), (GOD, PER, -1.0), (GOD, ZG, -1.0)]
# chunks of 124 and 120 cells, blocks of four of them, one block of twelve, then several
SIZES = [9, 16, 17, 119, 120, 121, 123, 124, 125, 127, 480, 482, 483, 496, 497, 499, 1440, 1441, 1443, 1488, 1489, 1491, 3001, 20011]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("flux,bc,alpha", FORMS)
def test_sizes(hh, dev, n, flux, bc, alpha):
    for k in (3, 2):
        same(grad(hh, dev, n, k, flux, bc, 3, 4, False, alpha), grad(hh, dev, n, k, flux, bc, 3, 4, True, alpha))


@pytest.mark.parametrize("n", [500, 2500])
@pytest.mark.parametrize("order,steps", [(1, 2), (1, 5), (2, 1), (2, 4), (3, 1)])
@pytest.mark.parametrize("k", [1, 2, 3])
def test_orders(hh, dev, n, order, steps, k):
    for flux, bc, alpha in FORMS:
        same(grad(hh, dev, n, k, flux, bc, order, steps, False, alpha),
             grad(hh, dev, n, k, flux, bc, order, steps, True, alpha))


# around 256 blocks of 4 chunks and of 8 (the largest that go back in one launch), and the largest that go forward in one
@pytest.mark.parametrize("n", [122881, 126976, 126979, 253952, 253955, 700001, 1 << 20, 1187328, 1350000, 1396736, 1400000])
@pytest.mark.parametrize("flux,bc,alpha", [(LF, PER, -1.0), (LF, ZG, -1.0), (GOD, ZG, -1.0)])
def test_large(hh, dev, n, flux, bc, alpha):
    same(grad(hh, dev, n, 3, flux, bc, 3, 2, False, alpha), grad(hh, dev, n, 3, flux, bc, 3, 2, True, alpha))


@pytest.mark.parametrize("n", [700, 1489, 5001])
@pytest.mark.parametrize("bc", [PER, ZG])
def test_maximum_at_block_ends_and_ties(hh, dev, n, bc):
    """The cell that takes alpha's cotangent at the ends of blocks and of the line, and several
    cells at the maximum (the first takes it)."""
    ch = 496 if bc == PER else 480
    spots = [[0], [1], [n - 1], [n - 2], [ch - 1], [ch], [ch + 2], [ch - 3], [3, n - 1], [ch - 1, ch], [5, ch + 1, n - 1]]
    for at in spots:
        u = 0.3 + 0.2 * np.sin(2 * math.pi * np.arange(n) / n)
        u[[j for j in at if j < n]] = -1.7
        same(grad(hh, dev, n, 3, LF, bc, 3, 2, False, u=u), grad(hh, dev, n, 3, LF, bc, 3, 2, True, u=u))


@pytest.mark.parametrize("n", [200, 40000])
@pytest.mark.parametrize("arith", ["fast", "exact"])
def test_many_passes_on_one_object(hh, dev, n, arith):
    same(grad(hh, dev, n, 3, LF, PER, 3, 6, False, arith=arith, reps=20), grad(hh, dev, n, 3, LF, PER, 3, 6, True, arith=arith))


@pytest.mark.parametrize("n", [3001, 30000])
@pytest.mark.parametrize("flux,bc", [(LF, PER), (LF, ZG), (GOD, ZG)])
def test_waits_in_vain_fall_back(hh, dev, monkeypatch, n, flux, bc):
    ref = grad(hh, dev, n, 3, flux, bc, 3, 5, True)
    monkeypatch.setenv("HRW_RESIDENT_POLLS", "1")
    same(grad(hh, dev, n, 3, flux, bc, 3, 5, False, reps=3), ref)


def test_recording_integrate_in_place(hh, dev):
    """rktvd's tape and adjoint: state and cotangent are replaced in place, also after a wait in vain."""
    import torch
    n, steps = 5000, 7
    u0, g, dt = case(n)
    out = []
    for tuned in (False, True):
        p = hh.Burgers1D(n)
        if tuned:
            p.tune(0, 4)
        ode = hh.RkTvd(p, order=3).tape(steps)
        u, lam = torch.as_tensor(u0, device=dev).clone(), torch.as_tensor(g, device=dev).clone()
        t = ode.integrate(u, 0.0, (steps - 0.5) * dt, dt)
        ode.adjoint(lam)
        out.append((u.cpu().numpy(), lam.cpu().numpy(), t))
    same(out[0], out[1])
    assert out[0][2] == out[1][2]


@pytest.mark.parametrize("value", [math.nan, math.inf])
@pytest.mark.parametrize("n", [300, 3001])
@pytest.mark.parametrize("bc", [PER, ZG])
def test_nonfinite_state(hh, dev, n, value, bc):
    u = case(n)[0].copy()
    u[n // 2] = value
    a, b = (grad(hh, dev, n, 3, LF, bc, 3, 3, tuned, u=u) for tuned in (False, True))
    assert np.array_equal(a[0], b[0], equal_nan=True) and np.array_equal(a[1], b[1], equal_nan=True)
