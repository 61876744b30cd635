"""Lines of a batch whose blocks wait for each other in vain (a few polls per wait) are computed anew in
the stream: the results are those of the launches per stage (set_cells_per_lane), bit for bit."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LF, GOD = 0, 1


def state(ns):
    out = []
    for i, n in enumerate(ns):
        rng = np.random.default_rng(i + n)
        x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
        out.append(0.4 + np.sin(math.pi * x + 0.1 * i) + 0.5 * (x > 0.2) + 0.05 * rng.standard_normal(n))
    return out


def both(hh, dev, ns, flux, alpha, steps, calls, us=None):
    import torch
    us = us or state(ns)
    dts = np.array([0.2 * (2.0 / n) / 2.5 for n in ns])
    res = []
    for fixed in (False, True):
        b = hh.BurgersBatch(ns, [1 + i % 3 for i in range(len(ns))], dts, flux=flux, alpha=alpha)
        if fixed:
            b.set_cells_per_lane(6)
        u = b.pack(us, dev)
        for _ in range(calls):
            b.step(u, steps)
        torch.cuda.synchronize()
        res.append((u.cpu().numpy(), b.t.copy()))
    assert np.array_equal(res[0][0], res[1][0], equal_nan=True) and np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("flux,alpha", [(LF, -1.0), (LF, 2.5), (GOD, -1.0)])
@pytest.mark.parametrize("polls", [0, 1, 20])
@pytest.mark.parametrize("steps,calls", [(3, 3), (66, 1)])
def test_waits_in_vain(hh, dev, monkeypatch, flux, alpha, polls, steps, calls):
    monkeypatch.setenv("HRW_RESIDENT_POLLS", str(polls))
    both(hh, dev, [3500, 110336, 5000, 40, 7001, 20000, 20001, 1500], flux, alpha, steps, calls)


def test_waits_in_vain_of_many_lines(hh, dev, monkeypatch):
    monkeypatch.setenv("HRW_RESIDENT_POLLS", "3")
    both(hh, dev, [6000 + 17 * i for i in range(300)], LF, -1.0, 2, 2)


def test_wait_in_vain_is_made_good_once(hh, dev, monkeypatch):
    """A later call whose waits are long enough goes on from it."""
    import torch
    ns = [5000, 9000]
    dts = np.array([1e-5, 1e-5])
    monkeypatch.setenv("HRW_RESIDENT_POLLS", "1")
    a = hh.BurgersBatch(ns, [3, 2], dts)
    monkeypatch.delenv("HRW_RESIDENT_POLLS")
    b = hh.BurgersBatch(ns, [3, 2], dts)
    u = a.pack(state(ns), dev)
    v = u.clone()
    for x in (a, b):
        x.step(u, 5)
        b.step(v, 5)
    torch.cuda.synchronize()
    assert torch.equal(u, v)


@pytest.mark.parametrize("value", [math.nan, math.inf])
def test_non_finite_line(hh, dev, monkeypatch, value):
    monkeypatch.setenv("HRW_RESIDENT_POLLS", "1")
    ns = [5000, 5000, 300]
    us = state(ns)
    us[1][77] = value
    both(hh, dev, ns, LF, -1.0, 2, 1, us)
