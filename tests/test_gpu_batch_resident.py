"""The batch's whole-integration kernel (the default) against its kernels per stage
(set_cells_per_lane selects those), bit for bit: lines at the edges of lanes, wavefronts and blocks,
lines split over blocks that exchange, every flux, many calls."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LF, GOD = 0, 1


def lines(ns, seed=1):
    rng = np.random.default_rng(seed)
    out = []
    for n in ns:
        x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
        out.append(0.5 + 0.4 * np.sin(math.pi * x + rng.uniform(0, 6)) + 0.3 * np.sin(2 * math.pi * x + rng.uniform(0, 6))
                   + 0.4 * (x > rng.uniform(-0.5, 0.5)) + 0.01 * rng.standard_normal(n))
    return out


def both(hh, dev, ns, ks, flux, alpha, steps, calls=1, graph=True):
    us = lines(ns)
    dts = np.array([0.25 * (2.0 / n) / max(0.1, np.abs(u).max()) for n, u in zip(ns, us)])
    res = []
    for fixed in (False, True):
        b = hh.BurgersBatch(ns, ks, dts, flux=flux, alpha=alpha)
        if fixed:
            b.set_cells_per_lane(6)
        u = b.pack(us, dev)
        for _ in range(calls):
            b.step(u, steps, graph=graph)
        import torch
        torch.cuda.synchronize()
        res.append((u.cpu().numpy(), b.t.copy()))
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])


FLUXES = [(LF, -1.0), (LF, 2.0), (GOD, -1.0)]


@pytest.mark.parametrize("flux,alpha", FLUXES)
@pytest.mark.parametrize("top", [2048, 9000])
def test_line_lengths(hh, dev, flux, alpha, top):
    """Two cells per lane (no line above 2048 cells) and four."""
    ns = [1, 2, 3, 5, 7, 8, 9, 61, 62, 63, 64, 123, 124, 125, 247, 248, 249, 991, 992, 993, 1723, 1724, 1735, 1736, 1737, 1983,
          1984, 1985, top]
    ns = [n for n in ns if n <= top]
    for k in (1, 2, 3):
        both(hh, dev, ns, [k] * len(ns), flux, alpha, 5)


@pytest.mark.parametrize("flux,alpha", FLUXES)
def test_split_lines(hh, dev, flux, alpha):
    """Lines over 2 to 64 blocks, with short ones between them; more blocks than the chip holds."""
    rng = np.random.default_rng(4)
    ns = [110336, 40000, 3448, 3449, 3473, 5000, 3970, 100, 17, 65536, 20001] + list(rng.integers(2000, 30000, 60))
    both(hh, dev, ns, [2 + i % 2 for i in range(len(ns))], flux, alpha, 3)


@pytest.mark.parametrize("n", [110337, 126209])
def test_lines_that_do_not_fit_take_the_stages(hh, dev, n):
    both(hh, dev, [n, 300], [3, 2], LF, -1.0, 2)


@pytest.mark.parametrize("graph", [True, False])
def test_many_calls_and_long_calls(hh, dev, graph):
    both(hh, dev, [300, 5000, 12000], [3, 3, 2], LF, -1.0, 3, calls=25, graph=graph)
    both(hh, dev, [300, 5000], [3, 2], LF, -1.0, 150, graph=graph)   # several launches in one call


def test_tune_keeps_bits(hh, dev):
    ns = [500, 3000, 9000]
    us = lines(ns)
    dts = np.full(3, 1e-5)
    b = hh.BurgersBatch(ns, [3, 2, 3], dts)
    u = b.pack(us, dev)
    b.step(u, 4)
    c = hh.BurgersBatch(ns, [3, 2, 3], dts)
    v = c.pack(us, dev)
    c.tune(v)
    c.step(v, 4)
    import torch
    torch.cuda.synchronize()
    assert torch.equal(u, v)


def test_two_batches_on_two_streams(hh, dev):
    import torch
    ns, ks = [30000, 20000, 700] * 20, [3, 2, 3] * 20
    us = lines(ns)
    dts = np.array([0.25 * (2.0 / n) / 2.0 for n in ns])
    bs = [hh.BurgersBatch(ns, ks, dts) for _ in range(2)]
    st = [torch.cuda.Stream() for _ in bs]
    us_d = [b.pack(us, dev) for b in bs]
    torch.cuda.synchronize()
    for _ in range(4):
        for b, s, u in zip(bs, st, us_d):
            with torch.cuda.stream(s):
                b.step(u, 3)
    torch.cuda.synchronize()
    ref = hh.BurgersBatch(ns, ks, dts)
    ref.set_cells_per_lane(6)
    v = ref.pack(us, dev)
    ref.step(v, 12)
    torch.cuda.synchronize()
    assert torch.equal(us_d[0], v) and torch.equal(us_d[1], v)


# an ensemble of many rounds (five cells per lane): lines at the edges of one block and of two
@pytest.mark.parametrize("flux,alpha", [(LF, -1.0), (LF, 2.5), (GOD, -1.0)])
def test_many_rounds(hh, dev, flux, alpha):
    ns = [61000] * 48 + [2151, 2152, 2153, 2479, 2480, 2481, 4304, 4305, 4306, 4944, 4945, 310, 311, 40, 5]
    assert sum(ns) > 2900000
    both(hh, dev, ns, [2 + i % 2 for i in range(len(ns))], flux, alpha, 3)
