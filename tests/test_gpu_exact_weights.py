"""EXACT arithmetic at the ends of its range: the quotients of the nonlinear weights that share a
reciprocal (sum of (eps + beta)^2 below 2^400) and the divides beyond it must both be the correctly
rounded quotients, hence the oracle's bits (numeric equality)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def states(n, seed):
    """Cells whose jumps lie far below, around and far beyond 2^100 (where the sum of squares of
    the indicators passes 2^400), mixed and apart."""
    rng = np.random.default_rng(seed)
    sign = rng.choice([-1.0, 1.0], n)
    yield sign * 10.0 ** rng.uniform(-150, -100, n)
    yield sign * 10.0 ** rng.uniform(-8, 8, n)
    yield sign * 2.0 ** rng.uniform(98, 102, n)
    yield sign * 10.0 ** rng.uniform(31, 60, n)
    yield sign * 10.0 ** rng.choice([-140.0, -3.0, 0.0, 29.0, 31.0, 55.0], n)
    yield np.where(np.arange(n) < n // 2, 1.0, 3.0)


@pytest.mark.parametrize("eps", [3e-16, 1e-6, 10.0])
@pytest.mark.parametrize("k", [2, 3])
def test_reconstruct_range(oracle, hh, dev, k, eps):
    import torch
    for v in states(777, 31 * k):
        t = torch.as_tensor(v, device=dev)
        vl, vr = hh.Weno(v.size, k, eps, arith="exact").reconstruct(t)
        ol, orr = oracle.reconstruct(v, k, eps)
        assert np.array_equal(vl.cpu().numpy(), ol) and np.array_equal(vr.cpu().numpy(), orr)


@pytest.mark.parametrize("n1,n2", [(61, 7), (130, 33)])
@pytest.mark.parametrize("k", [2, 3])
def test_pbe_rhs_range(oracle, hh, dev, k, n1, n2):
    import torch
    e1 = oracle.grid_linear(0.0, 1.0, n1)
    e2 = oracle.grid_linear(0.0, 1.0, n2)
    for v in states(n1 * n2, 7 * k):
        p = hh.PBE2D(n1, n2, k, 1e-6, bc=hh.BC_INFLOW0_OUTFLOW, arith="exact")
        got = p.rhs(0.0, torch.as_tensor(v, device=dev)).cpu().numpy()
        ref = oracle.pbe_rhs(v, e1, e2, k=k, bc=1)
        assert np.array_equal(got, ref)
