"""The three kernels of the many-lines reconstruction (one or two cells per thread along the line,
wavefronts across strided lines) against the oracle line by line: EXACT and non-uniform lines bit
for bit, FAST to 1e-12 of max|v|; what lies between the lines stays untouched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(oracle, hh, dev, n, nlines, incv, ldv, inco, ldo, k, arith, xedges=None, every=1):
    import torch
    rng = np.random.default_rng(n * 1000 + nlines)
    size = (nlines - 1) * ldv + (n - 1) * incv + 1
    osize = (nlines - 1) * ldo + (n - 1) * inco + 1
    v = rng.standard_normal(size)
    d = torch.as_tensor(v, device=dev)
    vl = torch.full((osize,), 7.0, dtype=torch.float64, device=dev)
    vr = torch.full((osize,), 7.0, dtype=torch.float64, device=dev)
    w = hh.Weno(n, k, 1e-6, xedges=xedges, arith=arith)
    w.reconstruct_lines(d, nlines, incv, ldv, vl, vr, inco, ldo)
    L, R = vl.cpu().numpy(), vr.cpu().numpy()
    cnu = None if xedges is None else oracle.calc_cnu(k, xedges)
    touched = np.zeros(osize, bool)
    i = np.arange(n)
    for l in range(nlines):
        touched[l * ldo + i * inco] = True
        if l % every and l != nlines - 1:
            continue
        ol, orr = oracle.reconstruct(v[l * ldv + i * incv].copy(), k, 1e-6, cnu=cnu)
        gl, gr = L[l * ldo + i * inco], R[l * ldo + i * inco]
        if arith == "exact" or xedges is not None:
            assert np.array_equal(gl, ol) and np.array_equal(gr, orr), (n, nlines, l)
        else:
            tol = 1e-12 * np.abs(v).max()
            assert np.abs(gl - ol).max() <= tol and np.abs(gr - orr).max() <= tol, (n, nlines, l)
    assert np.all(L[~touched] == 7.0) and np.all(R[~touched] == 7.0)


@pytest.mark.parametrize("n,nlines", [(1, 8), (2, 64), (7, 63), (8, 65), (9, 7), (31, 130), (32, 8),
                                      (33, 129), (100, 250)])
@pytest.mark.parametrize("k,arith", [(1, "exact"), (2, "exact"), (3, "exact"), (2, "fast"), (3, "fast")])
def test_across(oracle, hh, dev, n, nlines, k, arith):
    check(oracle, hh, dev, n, nlines, nlines, 1, nlines, 1, k, arith)                # packed
    check(oracle, hh, dev, n, nlines, 2 * nlines + 3, 2, 3 * nlines + 1, 3, k, arith)    # gaps


@pytest.mark.parametrize("k", [1, 2, 3])
def test_across_nonuniform(oracle, hh, dev, k):
    xe = np.cumsum(np.random.default_rng(k).uniform(0.1, 1.0, 42))
    check(oracle, hh, dev, 41, 70, 70, 1, 70, 1, k, "fast", xedges=xe)


def test_mixed_directions(oracle, hh, dev):
    """Strided lines in, contiguous lines out, and the other way round."""
    check(oracle, hh, dev, 40, 30, 30, 1, 1, 40, 3, "exact")
    check(oracle, hh, dev, 40, 30, 1, 40, 30, 1, 3, "exact")


@pytest.mark.parametrize("arith", ["exact", "fast"])
@pytest.mark.parametrize("n,nlines,ld", [(512, 1024, 512), (1031, 520, 1033), (1537, 350, 1537)])
def test_two_cells_per_thread(oracle, hh, dev, n, nlines, ld, arith):
    check(oracle, hh, dev, n, nlines, 1, ld, 1, ld, 3, arith, every=97)
