"""The work whose speed is measured: integrations, gradients and reconstructions as programs call
them through the Python mirror (hr-weno_amd/hrweno_hip), from the 100-cell line of the first
example to a line of 2**24 cells, with inputs drawn from a seed.

Kinds of case (the field "kind"):
  line     RkTvd / MsTvd.integrate of one 1D Burgers line, either flux, either kind of ends,
           both arithmetic forms, linear or non-uniform grid
  pbe      the same of the 2D population balance (the second example)
  batch    BurgersBatch.step of an uneven ensemble of periodic lines
  adjoint  a forward and backward through autograd.evolve (or, for the multistep method,
           tape / integrate / adjoint)
  sweeps   the reconstructions of example 2's right-hand side: every x1 line (contiguous) and
           every x2 line (strided) of one 2D state, one call each
  rhs      one right-hand side evaluation of a line (a user's own integrator, or steady-state
           residual)

`exact` restates the scheme in plain torch float64 in the textbook order.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hr-weno_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import hrweno_hip as hh                                    # noqa: E402
from hrweno_hip.autograd import evolve                     # noqa: E402

EPS = 1e-6
CFL = 0.4


def listed():
    return [
        # the first example as it stands: 100 cells, Godunov flux, zero-gradient ends, one output
        # interval (12 RK3 steps) per call: the smallest call, all launches and latency
        {"name": "example1_100", "kind": "line", "n": 100, "steps": 12, "flux": "godunov",
         "bc": "zerograd", "arith": "fast", "method": "rk3", "k": 3, "grid": "linear"},
        # a teaching- or validation-size periodic line with the Lax-Friedrichs flux, a whole run's
        # worth of steps
        {"name": "line_1000", "kind": "line", "n": 1000, "steps": 200, "flux": "lf",
         "bc": "periodic", "arith": "fast", "method": "rk3", "k": 3, "grid": "linear"},
        # an ordinary production line, of no round size
        {"name": "line_50021", "kind": "line", "n": 50021, "steps": 60, "flux": "lf",
         "bc": "periodic", "arith": "fast", "method": "rk3", "k": 3, "grid": "linear"},
        # example 1's composition on a fine grid of no round size
        {"name": "godunov_1000003", "kind": "line", "n": 1000003, "steps": 40, "flux": "godunov",
         "bc": "zerograd", "arith": "fast", "method": "rk3", "k": 3, "grid": "linear"},
        # the benchmark's headline line
        {"name": "line_2p24", "kind": "line", "n": 1 << 24, "steps": 6, "flux": "lf",
         "bc": "periodic", "arith": "fast", "method": "rk3", "k": 3, "grid": "linear"},
        # a run that has to match the reference bit for bit
        {"name": "exact_300007", "kind": "line", "n": 300007, "steps": 30, "flux": "lf",
         "bc": "periodic", "arith": "exact", "method": "rk3", "k": 3, "grid": "linear"},
        # a stretched grid (reconstruction coefficients of its own in every cell)
        {"name": "stretched_60001", "kind": "line", "n": 60001, "steps": 30, "flux": "godunov",
         "bc": "zerograd", "arith": "fast", "method": "rk3", "k": 3, "grid": "stretched"},
        # the second example at its own size, one output interval (10 steps) after the start
        {"name": "pbe_250", "kind": "pbe", "n1": 250, "n2": 250, "steps": 14, "bc": "zeroflux",
         "arith": "fast", "method": "ms", "k": 3},
        # the benchmark's 2D workload in the form it is quoted in
        {"name": "pbe_exact_2048", "kind": "pbe", "n1": 2048, "n2": 2048, "steps": 16,
         "bc": "outflow", "arith": "exact", "method": "rk3", "k": 3},
        # an uneven ensemble, lengths log-uniform in [256, 65536], orders mixed
        {"name": "batch_1024", "kind": "batch", "lines": 1024, "lo": 256, "hi": 65536, "steps": 6,
         "flux": "lf", "k": 0},
        # the gradient of a benchmark-size line with respect to its initial data
        {"name": "adjoint_2p20", "kind": "adjoint", "n": 1 << 20, "steps": 20, "flux": "lf",
         "bc": "periodic", "method": "rk3", "k": 3},
        # both sweeps of a 2D state, as example 2's own right-hand side calls reconstruct
        {"name": "sweeps_1500x1200", "kind": "sweeps", "n1": 1500, "n2": 1200, "arith": "fast",
         "k": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above; odd sizes come up by themselves."""
    kind = rng.choice(["line"] * 5 + ["pbe"] * 2 + ["batch"] * 2 + ["adjoint"] * 3 +
                      ["sweeps"] * 2 + ["rhs"])
    k = rng.choice([3, 3, 3, 2])
    if kind == "line":
        grid = rng.choice(["linear"] * 4 + ["stretched"])
        arith = rng.choice(["fast", "fast", "exact"])
        if grid == "stretched":
            n = _log_int(rng, 100, 200_000)
        elif arith == "exact":
            n = _log_int(rng, 100, 2_000_000)
        else:
            n = _log_int(rng, 100, 8_000_000)
        # (the multistep method amplifies rounding, so its runs are short ones)
        method = rng.choice(["rk3", "rk3", "rk2", "rk1", "ms"])
        most = 16 if method == "ms" else 40 if method == "rk1" else 200
        return {"kind": kind, "n": n, "steps": max(5, min(rng.randint(6, most), 30_000_000 // n)),
                "flux": rng.choice(["lf", "lf", "godunov"]),
                "bc": "zerograd" if grid == "stretched" else rng.choice(["periodic", "zerograd"]),
                "arith": arith, "method": method, "k": k, "grid": grid}
    if kind == "pbe":
        n1, n2 = _log_int(rng, 40, 1600), _log_int(rng, 40, 1600)
        return {"kind": kind, "n1": n1, "n2": n2,
                "steps": max(5, min(rng.randint(6, 40), 16_000_000 // (n1 * n2))),
                "bc": rng.choice(["outflow", "zeroflux"]), "arith": rng.choice(["fast", "exact"]),
                "method": rng.choice(["rk3", "ms"]), "k": k}
    if kind == "batch":
        lo = _log_int(rng, 64, 2048)
        return {"kind": kind, "lines": _log_int(rng, 8, 800), "lo": lo,
                "hi": _log_int(rng, 2 * lo, 65536), "steps": rng.randint(2, 12),
                "flux": rng.choice(["lf", "lf", "godunov"]), "k": 0}
    if kind == "adjoint":
        n = _log_int(rng, 200, 600_000)
        return {"kind": kind, "n": n, "steps": max(6, min(rng.randint(6, 16), 6_000_000 // n)),
                "flux": rng.choice(["lf", "godunov"]), "bc": rng.choice(["periodic", "zerograd"]),
                "method": rng.choice(["rk3", "rk3", "ms"]), "k": k}
    if kind == "sweeps":
        return {"kind": kind, "n1": _log_int(rng, 30, 1800), "n2": _log_int(rng, 30, 1500),
                "arith": rng.choice(["fast", "fast", "exact"]), "k": k}
    return {"kind": "rhs", "n": _log_int(rng, 100, 8_000_000), "flux": rng.choice(["lf", "godunov"]),
            "bc": rng.choice(["periodic", "zerograd"]), "arith": rng.choice(["fast", "exact"]),
            "k": k}


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator()
    g.manual_seed(seed)
    return g


def _rand(g, count, lo=0.0, hi=1.0):
    return (lo + (hi - lo) * torch.rand(count, generator=g, dtype=torch.float64)).tolist()


def _mean(case):
    """The waves' mean: transonic for Lax-Friedrichs; for the endpoint Godunov flux, which is no
    monotone flux at a sonic point, a state that keeps its sign."""
    return 2.5 if case["flux"] == "godunov" else 0.5


def _profile(x, g, mean, jumps=True):
    """A smooth wave of four modes about a mean, with (on request) three jumps."""
    amp, phi = _rand(g, 4, 0.1, 0.5), _rand(g, 4, 0.0, 2 * math.pi)
    u = torch.full_like(x, mean)
    for m in range(4):
        u += amp[m] / (m + 1) * torch.sin(math.pi * (m + 1) * x + phi[m])
    if jumps:
        for xj, hj in zip(_rand(g, 3, -0.9, 0.9), _rand(g, 3, -0.4, 0.4)):
            u += hj * (x >= xj)
    return u


def _widths(n, lo, hi, dev):
    """Cell widths of the linear grid as its edges lo + rx*i give them."""
    e = lo + torch.arange(n + 1, dtype=torch.float64, device=dev) * ((hi - lo) / n)
    return e[1:] - e[:-1]


def _centres(n, dev):
    return -1.0 + (torch.arange(n, dtype=torch.float64, device=dev) + 0.5) * (2.0 / n)


def _stretched_edges(n, g):
    """n+1 edges on [-1, 1], smoothly clustered about a seeded place."""
    s = torch.arange(n + 1, dtype=torch.float64) * (2.0 / n) - 1.0
    a, p = _rand(g, 1, 0.1, 0.25)[0], _rand(g, 1, 0.0, 2 * math.pi)[0]
    e = s + a / math.pi * (torch.sin(math.pi * s + p) - math.sin(-math.pi + p))
    return e


def _line_inputs(case, seed, dev):
    g = _gen(seed)
    n = case["n"]
    edges = None
    if case.get("grid") == "stretched":
        edges = _stretched_edges(n, g)
        x = ((edges[:-1] + edges[1:]) / 2).to(dev)
        dx = float((edges[1:] - edges[:-1]).min())
    else:
        x, dx = _centres(n, dev), 2.0 / n
    u0 = _profile(x, g, _mean(case), jumps=case["kind"] != "adjoint")
    return u0, edges, CFL * dx / float(u0.abs().max())


def _pbe_inputs(case, seed, dev):
    g = _gen(seed)
    n1, n2 = case["n1"], case["n2"]
    c1, c2, s = _rand(g, 1, 0.2, 0.4)[0], _rand(g, 1, 0.2, 0.4)[0], _rand(g, 1, 0.05, 0.1)[0]
    x1 = (torch.arange(n1, dtype=torch.float64, device=dev) + 0.5) / n1
    x2 = (torch.arange(n2, dtype=torch.float64, device=dev) + 0.5) / n2
    u0 = torch.exp(-((x1[None, :] - c1) ** 2 + (x2[:, None] - c2) ** 2) / (2 * s * s))
    return u0.reshape(-1).contiguous(), CFL / (1.5 * n1 + 0.5 * n2)


def _batch_sizes(case, seed):
    """Lengths, orders: a property of the case (the ensemble is the plan); data come from seed."""
    g = _gen(case["lines"] * 1000003 + case["lo"] * 31 + case["hi"])
    r = torch.rand(case["lines"], generator=g, dtype=torch.float64)
    n = torch.exp(math.log(case["lo"]) + r * math.log(case["hi"] / case["lo"])).round().to(torch.int64)
    k = 2 + (torch.rand(case["lines"], generator=g) < 0.5).to(torch.int64)
    return n, k


def _batch_inputs(case, seed, dev):
    n, k = _batch_sizes(case, seed)
    L = case["lines"]
    g = _gen(seed)
    nd = n.to(dev)
    line = torch.repeat_interleave(torch.arange(L, device=dev), nd)
    first = torch.cumsum(nd, 0) - nd
    i = torch.arange(line.numel(), device=dev) - first[line]
    x = -1.0 + (i.to(torch.float64) + 0.5) * (2.0 / nd.to(torch.float64))[line]

    def per_line(lo, hi):
        return (lo + (hi - lo) * torch.rand(L, generator=g, dtype=torch.float64)).to(dev)[line]
    u = per_line(-0.2, 0.1) + _mean(case)
    for m in range(3):
        u = u + per_line(0.1, 0.4) / (m + 1) * torch.sin(math.pi * (m + 1) * x + per_line(0.0, 2 * math.pi))
    u = u + per_line(-0.5, 0.5) * (x >= per_line(-0.6, 0.6))
    umax = torch.zeros(L, dtype=torch.float64, device=dev).scatter_reduce(0, line, u.abs(), "amax")
    dt = CFL * (2.0 / nd.to(torch.float64)) / umax
    return n, k, line, i, u, dt


_FLUX = {"lf": hh.LAX_FRIEDRICHS, "godunov": hh.GODUNOV}
_BC = {"periodic": hh.BC_PERIODIC, "zerograd": hh.BC_ZERO_GRADIENT, "zeroflux": hh.BC_ZERO_FLUX,
       "outflow": hh.BC_INFLOW0_OUTFLOW}
_ORDER = {"rk1": 1, "rk2": 2, "rk3": 3}


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    s = {"case": case}
    if kind in ("line", "rhs", "adjoint"):
        u0, edges, dt = _line_inputs(case, seed, dev)
        s.update(u0=u0, dt=dt, u=torch.empty_like(u0))
        s["problem"] = hh.Burgers1D(
            case["n"], k=case["k"], eps=EPS, flux=_FLUX[case["flux"]], bc=_BC[case["bc"]],
            arith=case.get("arith", "fast"), xedges=None if edges is None else edges.numpy())
        if kind == "line" and case["method"] != "ms":
            s["ode"] = hh.RkTvd(s["problem"], order=_ORDER[case["method"]])
        if kind == "adjoint":
            s["g"] = _profile(_centres(case["n"], dev), _gen(seed + 7919), 0.0, jumps=False)
            if case["method"] != "ms":
                s["adj"] = hh.Adjoint(s["problem"], nsteps=case["steps"], dt=dt)
    elif kind == "pbe":
        u0, dt = _pbe_inputs(case, seed, dev)
        s.update(u0=u0, dt=dt, u=torch.empty_like(u0))
        s["problem"] = hh.PBE2D(case["n1"], case["n2"], k=case["k"], eps=EPS, bc=_BC[case["bc"]],
                                arith=case["arith"])
        if case["method"] != "ms":
            s["ode"] = hh.RkTvd(s["problem"], order=_ORDER[case["method"]])
    elif kind == "batch":
        n, k, line, i, u, dt = _batch_inputs(case, seed, dev)
        s["batch"] = hh.BurgersBatch(n.numpy(), k.numpy(), dt.cpu().numpy(), eps=EPS,
                                     flux=_FLUX[case["flux"]])
        off = torch.as_tensor(s["batch"].offsets[:-1], device=dev)
        s["u0"] = torch.zeros(s["batch"].total, dtype=torch.float64, device=dev)
        s["u0"][off[line] + i] = u
        s["u"] = torch.empty_like(s["u0"])
    else:
        g = torch.Generator(device=dev)
        g.manual_seed(seed)
        n1, n2 = case["n1"], case["n2"]
        u0, _ = _pbe_inputs(case, seed, dev)
        s["v"] = u0 + 0.01 * torch.rand(n1 * n2, generator=g, dtype=torch.float64, device=dev)
        s["out"] = [torch.empty_like(s["v"]) for _ in range(4)]
        s["w1"] = hh.Weno(n1, k=case["k"], eps=EPS, arith=case["arith"])
        s["w2"] = hh.Weno(n2, k=case["k"], eps=EPS, arith=case["arith"])
    return s


# ------------------------------------------------------------------------------ the pass
def _tout(case, dt):
    return (case["steps"] - 0.5) * dt      # the loop control then takes exactly `steps` steps


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("line", "pbe"):
        # a run from its initial data: the multistep method's object is made for it (its history
        # starts with the run), a Runge-Kutta object serves every run
        ode = s["ode"] if "ode" in s else hh.MsTvd(s["problem"])
        u = s["u"].copy_(s["u0"])
        t = ode.integrate(u, 0.0, _tout(case, s["dt"]), s["dt"])
        return u, t
    if kind == "rhs":
        return s["problem"].rhs(0.0, s["u0"], s["u"])
    if kind == "batch":
        u = s["u"].copy_(s["u0"])
        s["batch"].step(u, case["steps"])
        return u
    if kind == "adjoint":
        if case["method"] == "ms":
            ode = hh.MsTvd(s["problem"]).tape(1)
            u = s["u"].copy_(s["u0"])
            ode.integrate(u, 0.0, _tout(case, s["dt"]), s["dt"])
            return u, ode.adjoint(s["g"].clone())
        u0 = s["u0"].detach().requires_grad_(True)
        uN = evolve(u0, s["adj"])
        (g0,) = torch.autograd.grad(uN, u0, s["g"])
        return uN.detach(), g0
    n1, n2, (l1, r1, l2, r2) = case["n1"], case["n2"], s["out"]
    s["w1"].reconstruct_lines(s["v"], n2, 1, n1, l1, r1, 1, n1)     # x1 lines (contiguous)
    s["w2"].reconstruct_lines(s["v"], n1, n1, 1, l2, r2, n1, 1)     # x2 lines (strided)
    return l1, r1, l2, r2


# ------------------------------------------------------------------------------ its work
_STAGES = {"rk1": 1, "rk2": 2, "rk3": 3, "ms": 1}
_RECON_FLOPS = {1: 2, 2: 40, 3: 90}        # candidates, indicators, weights of both faces
_FLUX_FLOPS = 14                           # flux, divergence, stage combination


def _stages(case):
    """Right-hand sides of an integration (the multistep method starts with four RK3 steps)."""
    if case["method"] == "ms":
        return 12 + max(0, case["steps"] - 4)
    return case["steps"] * _STAGES[case["method"]]


def work(case):
    kind = case["kind"]
    if kind == "batch":
        n, k = _batch_sizes(case, 0)
        cells = int(n.sum())
        per = sum(int(m) * (_RECON_FLOPS[int(q)] + _FLUX_FLOPS) for m, q in zip(n, k))
        return {"bytes": 16.0 * cells, "flops": 3.0 * case["steps"] * per}
    rec = _RECON_FLOPS[case["k"]]
    if kind == "sweeps":
        n = case["n1"] * case["n2"]
        return {"bytes": 40.0 * n, "flops": 2.0 * n * rec}
    if kind == "pbe":
        n = case["n1"] * case["n2"]
        return {"bytes": 16.0 * n, "flops": float(n) * _stages(case) * 2 * (rec + _FLUX_FLOPS)}
    n = case["n"]
    if kind == "rhs":
        return {"bytes": 16.0 * n, "flops": float(n) * (rec + _FLUX_FLOPS)}
    per = rec + _FLUX_FLOPS
    if kind == "adjoint":                  # the forward, and a reverse of about three times it
        return {"bytes": 32.0 * n, "flops": 4.0 * n * _stages(case) * per}
    b = 16.0 * n
    if case["grid"] == "stretched":
        b += 8.0 * (n + 1)
    return {"bytes": b, "flops": float(n) * _stages(case) * per}


# ------------------------------------------------------------------------------ plain float64
_C = {2: [[1.5, -0.5], [0.5, 0.5], [-0.5, 1.5]],
      3: [[11 / 6, -7 / 6, 1 / 3], [1 / 3, 5 / 6, -1 / 6], [-1 / 6, 5 / 6, 1 / 3],
          [1 / 3, -7 / 6, 11 / 6]]}
_D = {2: [2 / 3, 1 / 3], 3: [0.3, 0.6, 0.1]}


def _recon(v, k, cnu=None):
    """Left and right face values from v(m), the state shifted to cell i+m."""
    if k == 1:
        return v(0), v(0)
    if k == 2:
        beta = [(v(1) - v(0)) ** 2, (v(0) - v(-1)) ** 2]
    else:
        beta = [13 / 12 * (v(0) - 2 * v(1) + v(2)) ** 2 + (3 * v(0) - 4 * v(1) + v(2)) ** 2 / 4,
                13 / 12 * (v(-1) - 2 * v(0) + v(1)) ** 2 + (v(-1) - v(1)) ** 2 / 4,
                13 / 12 * (v(-2) - 2 * v(-1) + v(0)) ** 2 + (v(-2) - 4 * v(-1) + 3 * v(0)) ** 2 / 4]
    c = _C[k] if cnu is None else cnu
    right = [sum(c[r + 1][j] * v(j - r) for j in range(k)) for r in range(k)]
    left = [sum(c[r][j] * v(j - r) for j in range(k)) for r in range(k)]
    q = [(EPS + b) ** 2 for b in beta]
    a = [_D[k][r] / q[r] for r in range(k)]
    b = [_D[k][k - 1 - r] / q[r] for r in range(k)]
    vr = sum(a[r] * right[r] for r in range(k)) / sum(a)
    vl = sum(b[r] * left[r] for r in range(k)) / sum(b)
    return vl, vr


def _cnu(edges, k):
    """Coefficients c(j, r, i) of Shu's eq. 2.20 on a non-uniform grid, extended linearly."""
    ng = k + 1
    n = edges.numel() - 1
    steps = torch.arange(1, ng + 1, dtype=torch.float64)
    lo = edges[0] - (edges[1] - edges[0]) * steps.flip(0)
    hi = edges[n] + (edges[n] - edges[n - 1]) * steps
    x = torch.cat([lo, edges, hi])

    def e(m):                              # edge i + 1/2 + m of cells i = 1..n
        return x[ng + 1 + m: ng + 1 + m + n]
    out = []
    for r in range(-1, k):
        row = []
        for j in range(k):
            s2 = 0.0
            for m in range(j + 1, k + 1):
                den = 1.0
                for l in range(k + 1):
                    if l != m:
                        den = den * (e(m - r - 1) - e(l - r - 1))
                s1 = 0.0
                for l in range(k + 1):
                    if l == m:
                        continue
                    p = 1.0
                    for q in range(k + 1):
                        if q not in (m, l):
                            p = p * (e(0) - e(q - r - 1))
                    s1 = s1 + p
                s2 = s2 + s1 / den
            row.append(s2 * (e(j - r) - e(j - r - 1)))
        out.append(row)
    return out


def _godunov(fm, fp, vm, vp):
    return torch.where(vm <= vp, torch.minimum(fm, fp), torch.maximum(fm, fp))


def _first_max(u):
    a = u.abs()
    return a[(a == a.max()).nonzero()[0, 0]]


def _line_rhs(case, u, width, cnu):
    n, k = u.numel(), case["k"]
    h = k + 1
    i = torch.arange(-h, n + h, device=u.device)
    ext = u[i % n if case["bc"] == "periodic" else i.clamp(0, n - 1)]

    def v(m):                              # cells -1 .. n (with their neighbours)
        return ext[h - 1 + m: h - 1 + m + n + 2]
    c = cnu
    if c is not None:
        c = [[torch.cat([q[:1], q, q[-1:]]) for q in row] for row in c]
    vl, vr = _recon(v, k, c)
    vm, vp = vr[:-1], vl[1:]               # interfaces 1/2 .. n+1/2
    fm, fp = vm * vm / 2, vp * vp / 2
    if case["flux"] == "godunov":
        f = _godunov(fm, fp, vm, vp)
    else:
        f = (fm + fp - _first_max(u) * (vp - vm)) / 2
    if case["bc"] == "zerograd":
        f = torch.cat([f[1:2], f[1:-1], f[-2:-1]]) if n > 1 else f[:1].expand(2)
    return -(f[1:] - f[:-1]) / width


def _pbe_rhs(case, u):
    n1, n2, k = case["n1"], case["n2"], case["k"]
    w = u.reshape(n2, n1)

    def sweep(axis, n, coef):
        h = k
        i = torch.arange(-h, n + h, device=u.device).clamp(0, n - 1)
        ext = w.index_select(axis, i)
        vl, vr = _recon(lambda m: ext.narrow(axis, h + m, n), k)
        e = torch.arange(1, n + 1, dtype=torch.float64, device=u.device) / n
        gr = coef[0] + coef[1] * e
        gr = gr[None, :] if axis == 1 else gr[:, None]
        vm, vp = vr.narrow(axis, 0, n - 1), vl.narrow(axis, 1, n - 1)
        gi = gr.narrow(axis, 0, n - 1)
        f = _godunov(gi * vm, gi * vp, vm, vp)
        zero = torch.zeros_like(w.narrow(axis, 0, 1))
        last = gr.narrow(axis, n - 1, 1) * vr.narrow(axis, n - 1, 1) if case["bc"] == "outflow" else zero
        f = torch.cat([zero, f, last], axis)
        width = _widths(n, 0.0, 1.0, u.device)
        return -(f.narrow(axis, 1, n) - f.narrow(axis, 0, n)) / (width[None, :] if axis == 1 else width[:, None])
    return (sweep(1, n1, (1.0, 0.5)) + sweep(0, n2, (0.5, 0.0))).reshape(-1)


def _rk(rhs, u, dt, order):
    if order == 1:
        return u + dt * rhs(u)
    if order == 2:
        a = u + dt * rhs(u)
        return (u + a + dt * rhs(a)) / 2
    a = u + dt * rhs(u)
    b = (3 * u + a + dt * rhs(a)) / 4
    return (u + 2 * b + 2 * dt * rhs(b)) / 3


def _evolve(case, rhs, u, dt):
    if case["method"] != "ms":
        for _ in range(case["steps"]):
            u = _rk(rhs, u, dt, _ORDER[case["method"]])
        return u
    hist = []
    for _ in range(4):
        hist.append((u, rhs(u)))
        u = _rk(rhs, u, dt, 3)
    for _ in range(max(0, case["steps"] - 4)):
        L = rhs(u)
        uo, lo = hist.pop(0)
        hist.append((u, L))
        u = (25 * u + 50 * dt * L + 7 * uo + 10 * dt * lo) / 32
    return u


def _time(case, dt):
    t = 0.0
    for _ in range(case["steps"]):
        t = t + dt
    return t


def exact(case, seed):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    kind = case["kind"]
    if kind in ("line", "rhs", "adjoint"):
        u0, edges, dt = _line_inputs(case, seed, dev)
        width, cnu = _widths(case["n"], -1.0, 1.0, dev), None
        if edges is not None:
            width = (edges[1:] - edges[:-1]).to(dev)
            cnu = [[q.to(dev) for q in row] for row in _cnu(edges, case["k"])]

        def rhs(u):
            return _line_rhs(case, u, width, cnu)
        if kind == "rhs":
            return rhs(u0)
        if kind == "line":
            return _evolve(case, rhs, u0, dt), _time(case, dt)
        g = _profile(_centres(case["n"], dev), _gen(seed + 7919), 0.0, jumps=False)
        if case["method"] == "ms":
            if case["n"] * _stages(case) > 30_000_000:
                return None
            u = u0.clone().requires_grad_(True)
            uN = _evolve(case, rhs, u, dt)
            (g0,) = torch.autograd.grad(uN, u, g)
            return uN.detach(), g0
        states = [u0]
        with torch.no_grad():
            for _ in range(case["steps"]):
                states.append(_rk(rhs, states[-1], dt, 3))
        for u in reversed(states[:-1]):    # one step's graph at a time
            u = u.clone().requires_grad_(True)
            (g,) = torch.autograd.grad(_rk(rhs, u, dt, 3), u, g)
        return states[-1], g
    if kind == "pbe":
        u0, dt = _pbe_inputs(case, seed, dev)
        return _evolve(case, lambda u: _pbe_rhs(case, u), u0, dt), _time(case, dt)
    if kind == "batch":
        n, k, line, i, u, dt = _batch_inputs(case, seed, dev)
        nd = n.to(dev)
        first = (torch.cumsum(nd, 0) - nd)[line]
        at = {m: first + (i + m) % nd[line] for m in range(-3, 4)}
        k2 = (k == 2).to(dev)[line]
        rx, h = (2.0 / nd.to(torch.float64))[line], dt[line]
        width = (-1.0 + rx * (i + 1)) - (-1.0 + rx * i)

        def brhs(u):
            def v(m):
                return u[at[m]]
            l2, r2 = _recon(v, 2)
            l3, r3 = _recon(v, 3)
            vl, vr = torch.where(k2, l2, l3), torch.where(k2, r2, r3)
            vm, vp = vr, vl[at[1]]         # interface i+1/2
            if case["flux"] == "godunov":
                f = _godunov(vm * vm / 2, vp * vp / 2, vm, vp)
            else:
                a = torch.zeros(case["lines"], dtype=torch.float64, device=dev)
                a = a.scatter_reduce(0, line, u.abs(), "amax")[line]
                f = (vm * vm / 2 + vp * vp / 2 - a * (vp - vm)) / 2
            return -(f - f[at[-1]]) / width
        for _ in range(case["steps"]):
            u = _rk(brhs, u, h, 3)
        pad = (nd + 31) // 32 * 32         # lines start on 256-byte boundaries in the flat state
        flat = torch.zeros(int(pad.sum()), dtype=torch.float64, device=dev)
        flat[(torch.cumsum(pad, 0) - pad)[line] + i] = u
        return flat
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    n1, n2, k = case["n1"], case["n2"], case["k"]
    u0, _ = _pbe_inputs(case, seed, dev)
    v = (u0 + 0.01 * torch.rand(n1 * n2, generator=g, dtype=torch.float64, device=dev)).reshape(n2, n1)
    out = []
    for axis, n in ((1, n1), (0, n2)):
        i = torch.arange(-k, n + k, device=dev).clamp(0, n - 1)
        ext = v.index_select(axis, i)
        out += [t.contiguous().reshape(-1) for t in _recon(lambda m: ext.narrow(axis, k + m, n), k)]
    return out[0], out[1], out[2], out[3]
