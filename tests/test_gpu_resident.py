"""The whole-integration kernel (one launch per integrate call, one block or several exchanging end
cells and maxima) against one launch per stage -- a problem tuned to a kernel (tune(0, 4)) takes
those -- bit for bit, at the edges of its splits into lanes, wavefronts and blocks."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER, ZG = 0, 1
LF, GOD = 0, 1


def u0(n, seed=3):
    rng = np.random.default_rng(seed + n)
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    return (0.4 + np.sin(math.pi * x + 0.3) + 0.3 * np.sin(3 * math.pi * x) + 0.5 * (x > 0.2)
            + 0.01 * rng.standard_normal(n))


def run(hh, dev, n, flux, bc, k, arith, order, steps, tuned, alpha=-1.0, xedges=None, calls=1):
    import torch
    p = hh.Burgers1D(n, k, 1e-6, flux=flux, bc=bc, alpha=alpha, arith=arith, xedges=xedges)
    if tuned:
        p.tune(0, 4)
    ode = hh.RkTvd(p, order=order)
    dx = 2.0 / n if xedges is None else float(np.min(np.diff(xedges)))
    dt = 0.2 * dx / 2.5
    u = torch.as_tensor(u0(n), device=dev).clone()
    t = 0.0
    for _ in range(calls):
        t = ode.integrate(u, t, t + (steps - 0.5) * dt, dt)
    return u.cpu().numpy(), t, ode.fevals, ode.istate


def same(a, b):
    assert np.array_equal(a[0], b[0]) and a[1:] == b[1:]


# one block: lanes (62), wavefronts, one or two cells per lane; then two blocks and more
SIZES = [8, 9, 61, 62, 63, 124, 125, 619, 620, 621, 622, 1000, 1116, 1117, 1488, 1489, 1490, 3001]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("flux,bc,alpha", [(LF, PER, -1.0), (LF, ZG, -1.0), (LF, PER, 2.5), (GOD, ZG, -1.0),
                                           (GOD, PER, -1.0)])
@pytest.mark.parametrize("arith", ["fast", "exact"])
def test_sizes(hh, dev, n, flux, bc, alpha, arith):
    a = run(hh, dev, n, flux, bc, 3, arith, 3, 7, False, alpha)
    same(a, run(hh, dev, n, flux, bc, 3, arith, 3, 7, True, alpha))


@pytest.mark.parametrize("n", [500, 1300, 20011])
@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("arith", ["fast", "exact"])
def test_orders(hh, dev, n, order, k, arith):
    for flux, bc in ((LF, PER), (GOD, ZG)):
        same(run(hh, dev, n, flux, bc, k, arith, order, 9, False),
             run(hh, dev, n, flux, bc, k, arith, order, 9, True))


# the steps of the split: 96 blocks of 7 wavefronts (one, two cells per lane), 160 of 12, 256 blocks
# of more, four cells per lane, and just past what fits
@pytest.mark.parametrize("n", [40512, 40513, 82177, 108033, 187393, 236161, 473089, 949248, 949249, 1012736, 1012737])
@pytest.mark.parametrize("flux,bc,arith", [(LF, PER, "fast"), (GOD, ZG, "fast"), (LF, ZG, "exact"), (GOD, PER, "exact")])
def test_large(hh, dev, n, flux, bc, arith):
    same(run(hh, dev, n, flux, bc, 3, arith, 3, 3, False), run(hh, dev, n, flux, bc, 3, arith, 3, 3, True))


@pytest.mark.parametrize("n", [40, 620, 621, 5000, 108033, 235009])
@pytest.mark.parametrize("flux", [LF, GOD])
@pytest.mark.parametrize("k,arith", [(2, "fast"), (3, "fast"), (3, "exact")])
def test_nonuniform(hh, dev, n, flux, k, arith):
    e = np.linspace(-1.0, 1.0, n + 1)
    e = e + 0.2 / math.pi * np.sin(math.pi * e)
    same(run(hh, dev, n, flux, ZG, k, arith, 3, 4, False, xedges=e),
         run(hh, dev, n, flux, ZG, k, arith, 3, 4, True, xedges=e))


@pytest.mark.parametrize("n", [100, 30000])
def test_many_calls_on_one_object(hh, dev, n):
    """Exchange numbers go on from call to call; results and counters are those of single calls."""
    same(run(hh, dev, n, LF, PER, 3, "fast", 3, 5, False, calls=40), run(hh, dev, n, LF, PER, 3, "fast", 3, 5, True, calls=40))


def test_exact_equals_oracle(oracle, hh, dev):
    import torch
    for n in (1000, 7001):
        u = u0(n)
        e = oracle.grid_linear(-1.0, 1.0, n)
        w = np.diff(e)
        dt = 0.2 * (2.0 / n) / 2.5
        d = torch.as_tensor(u, device=dev).clone()
        hh.RkTvd(hh.Burgers1D(n, arith="exact"), order=3).integrate(d, 0.0, 49.5 * dt, dt)
        ref, _, steps, _ = oracle.burgers_rk(u, w, tout=49.5 * dt, dt=dt)
        assert steps == 50 and np.array_equal(d.cpu().numpy(), ref)


@pytest.mark.parametrize("n", [200, 50000])
def test_nonfinite_state_is_reported_and_cleared(hh, dev, n):
    import torch
    p = hh.Burgers1D(n)
    dt = 1e-3 / n
    bad = torch.as_tensor(u0(n), device=dev).clone()
    bad[n // 2] = float("nan")
    ode = hh.RkTvd(p, order=3)
    with pytest.raises(hh.HrwError, match="non-finite"):
        ode.integrate(bad, 0.0, 4.5 * dt, dt)
    assert ode.istate == -1
    good = hh.RkTvd(p, order=3)
    u = torch.as_tensor(u0(n), device=dev).clone()
    good.integrate(u, 0.0, 4.5 * dt, dt)
    assert bool(torch.isfinite(u).all())


@pytest.mark.parametrize("n", [300, 40000])
def test_two_objects_on_two_streams(hh, dev, n):
    """Objects share nothing: interleaved calls on two streams give what each gives alone."""
    import torch
    ref = run(hh, dev, n, LF, PER, 3, "fast", 3, 6, False, calls=5)[0]
    p = hh.Burgers1D(n)
    dt = 0.2 * (2.0 / n) / 2.5
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    odes = [hh.RkTvd(p, order=3) for _ in streams]
    us = [torch.as_tensor(u0(n), device=dev).clone() for _ in streams]
    ts = [0.0, 0.0]
    torch.cuda.synchronize()
    for _ in range(5):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                ts[i] = odes[i].integrate(us[i], ts[i], ts[i] + 5.5 * dt, dt)
    torch.cuda.synchronize()
    for u in us:
        assert np.array_equal(u.cpu().numpy(), ref)


@pytest.mark.parametrize("n", [3001, 30000])
@pytest.mark.parametrize("flux,bc", [(LF, PER), (GOD, ZG)])
def test_waits_in_vain_fall_back(hh, dev, monkeypatch, n, flux, bc):
    """Blocks that wait in vain (one poll per wait) leave the state as it was, and the call goes on
    with one launch per stage."""
    ref = run(hh, dev, n, flux, bc, 3, "fast", 3, 8, True, calls=3)
    monkeypatch.setenv("HRW_RESIDENT_POLLS", "1")
    same(run(hh, dev, n, flux, bc, 3, "fast", 3, 8, False, calls=3), ref)


def test_threads(hh, dev):
    """Integrations of several threads at once, each on a stream of its own (one of them at a time
    takes the exchanging kernel)."""
    import threading

    import torch
    n = 40000
    ref = run(hh, dev, n, LF, PER, 3, "fast", 3, 6, True, calls=8)[0]
    p = hh.Burgers1D(n)
    dt = 0.2 * (2.0 / n) / 2.5
    out = {}

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            ode = hh.RkTvd(p, order=3)
            u = torch.as_tensor(u0(n), device=dev).clone()
            t = 0.0
            for _ in range(8):
                t = ode.integrate(u, t, t + 5.5 * dt, dt)
            s.synchronize()
            out[i] = u.cpu().numpy()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert len(out) == 3 and all(np.array_equal(v, ref) for v in out.values())


# five and eight cells per lane (Lax-Friedrichs, Godunov), and just past what fits
@pytest.mark.parametrize("n", [786433, 1187328, 1187329, 1266688, 1266689, 1393664, 1393665, 1520640, 1520641])
@pytest.mark.parametrize("flux,bc,k", [(LF, PER, 3), (GOD, ZG, 3), (LF, ZG, 2), (GOD, PER, 1)])
def test_largest(hh, dev, n, flux, bc, k):
    same(run(hh, dev, n, flux, bc, k, "fast", 3, 2, False), run(hh, dev, n, flux, bc, k, "fast", 3, 2, True))


@pytest.mark.parametrize("value", [math.nan, math.inf, -math.inf])
@pytest.mark.parametrize("n", [300, 5000])
def test_nonfinite_line_of_a_batch(hh, dev, n, value):
    """A line with a non-finite cell gives what the launches per stage give; its neighbours are untouched."""
    us = [u0(n), u0(n), u0(n)]
    us[1][n // 3] = value
    out = []
    for per_line in (False, True):
        b = hh.BurgersBatch(np.array([n, n, n]), np.array([3, 3, 3]), np.full(3, 1e-3 / n))
        u = b.pack(us, dev)
        (b.step_per_line if per_line else b.step)(u, 2)
        out.append(b.unpack(u))
    for x, y in zip(*out):
        assert np.array_equal(x, y, equal_nan=True)
    assert not np.isfinite(out[0][1]).all() and np.isfinite(out[0][0]).all() and np.array_equal(out[0][0], out[0][2])


# alpha's seed: one block of 1024 threads, and the launches past its range
@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 4097, 32767, 32768, 32769])
@pytest.mark.parametrize("at", [0, -1])
def test_seeded_maximum(hh, dev, n, at):
    """The right-hand side with alpha = max|u| is that with the maximum given as a fixed alpha."""
    import torch
    u = u0(n)
    u[at] = -4.0
    d = torch.as_tensor(u, device=dev)
    a, b = (torch.empty_like(d) for _ in range(2))
    hh.Burgers1D(n).rhs(0.0, d, a)
    hh.Burgers1D(n, alpha=4.0).rhs(0.0, d, b)
    assert torch.equal(a, b)
