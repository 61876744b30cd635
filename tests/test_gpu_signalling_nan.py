"""alpha = max|u| of a state that holds signalling NaNs is the maximum of its other cells, in the
whole-integration kernels as in the launches per stage."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def state(n, total=0):
    """The largest cell first, then NaNs in the cells that the same lanes read after it."""
    x = (np.arange(n) + 0.5) * (2.0 / n) - 1.0
    u = np.zeros(max(n, total))
    u[:n] = 0.5 + 0.4 * np.sin(3 * x)
    u[10] = -4.0
    u.view(np.uint64)[74:n:64] = 0x7ff0000000000001
    return u


def device(u, dev):
    """(bit for bit: arithmetic on the way would quiet the NaNs)"""
    import torch
    return torch.from_numpy(u.view(np.int64)).to(dev).view(torch.float64)


@pytest.mark.parametrize("n", [300, 5000])
def test_batch(hh, dev, n):
    out = []
    for fixed in (False, True):
        b = hh.BurgersBatch([n], [3], np.array([1e-3 / n]))
        if fixed:
            b.set_cells_per_lane(6)
        u = device(state(n, b.total), dev)
        b.step(u, 1)
        out.append(u.cpu().numpy()[:n])
    assert np.isnan(out[0]).any() and np.isfinite(out[0]).sum() > n // 4
    assert np.array_equal(out[0], out[1], equal_nan=True)


@pytest.mark.parametrize("n", [300, 5000])
def test_recorded_forward(hh, dev, n):
    import torch
    out = []
    for tuned in (False, True):
        p = hh.Burgers1D(n)
        if tuned:
            p.tune(0, 4)
        a = hh.Adjoint(p, nsteps=1, dt=1e-3 / n, ckpt_every=1)
        out.append(a.forward(device(state(n), dev)).cpu().numpy())
    torch.cuda.synchronize()
    assert np.isfinite(out[0]).sum() > n // 4
    assert np.array_equal(out[0], out[1], equal_nan=True)
