"""Timed workloads of the library: what a program built on it calls, over the
range of grids, backends and precisions it is used with.

Kinds of case (key "kind"):

  apply       ``ContactSolver.matvec_device``: one elastic response u = S p of
              a pressure field resident in HBM. Free space ("fft") or
              periodic, FP64 or FP32, any grid side.
  build       a new ``ContactSolver`` and its first response: what every change
              of grid, domain or modulus costs.
  tangential  ``TangentialFFTOperator.matvec_device``: the shear response.
  solve       ``ContactSolver.solve`` on one grid, host arrays in and out.
  nested      ``solve_nested_device``: coarse-to-fine solve of a gap in HBM.
  adjoint     ``ContactSolver.adjoint_device``: gradient of a loss on the
              pressure of a converged solve with respect to the gap.
  ensemble    ``solve_ensemble_device``: independent solves advanced together.

Solves run in FP64 to a tolerance at which rounding alone hardly moves the
fields they return (1e-13); single precision is in the responses, which are
what such a solve spends its time on.
"""
import math

import numpy as np
import torch

from aspher_amd import api
from aspher_amd.tangential import TangentialFFTOperator

SOLVE_TOL = 1e-12


def listed():
    return [
        # the smallest grid a nested solve or a parameter study works on: the
        # call is launches and waits
        dict(name="apply_fft_64_f64", kind="apply", backend="fft", Ns=64, bits=64),
        # an ordinary free-space grid in single precision
        dict(name="apply_fft_512_f32", kind="apply", backend="fft", Ns=512, bits=32),
        # certification and refinement of a large free-space solve
        dict(name="apply_fft_2048_f64", kind="apply", backend="fft", Ns=2048, bits=64),
        # the largest free-space grid: the single-precision stage of the
        # mixed 4096^2 solve is this call, hundreds of times over
        dict(name="apply_fft_4096_f32", kind="apply", backend="fft", Ns=4096, bits=32),
        # periodic surfaces in double precision
        dict(name="apply_periodic_2048_f64", kind="apply", backend="periodic", Ns=2048, bits=64),
        # measured topographies come with the sides their instrument gives:
        # round decimal numbers, free space
        dict(name="apply_fft_1000_f64", kind="apply", backend="fft", Ns=1000, bits=64),
        # ... and an odd side on the torus
        dict(name="apply_periodic_1215_f32", kind="apply", backend="periodic", Ns=1215, bits=32),
        # a new solver for a new material or domain size
        dict(name="build_fft_1024", kind="build", backend="fft", Ns=1024, bits=64),
        # shear response in a friction loop
        dict(name="tangential_512_f64", kind="tangential", Ns=512, bits=64),
        # one small certified solve: hundreds of short kernels
        dict(name="solve_fft_256", kind="solve", backend="fft", Ns=256, precond="fourier",
             p_nominal=0.005),
        # a nested solve with the active set: coarse levels from 64^2 up, the
        # stencil preconditioner
        dict(name="nested_fft_1024", kind="nested", backend="fft", Ns=1024, engine="auto",
             active=True, p_nominal=0.005),
        # backward pass of a solve, periodic
        dict(name="adjoint_periodic_512", kind="adjoint", backend="periodic", Ns=512,
             p_nominal=0.01),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A grid side in [lo, hi]: powers of two, round decimal numbers, and any
    integer, odd ones and primes among them."""
    how = rng.random()
    if how < 0.4:
        a, b = math.ceil(math.log2(lo)), math.floor(math.log2(hi))
        return 1 << rng.randint(a, b)
    v = _log_int(rng, lo, min(hi, 2047))
    if how < 0.7:
        step = 10 if v < 400 else 50
        return max(lo, v // step * step)
    return v


def draw(rng):
    """Backends, precisions and preconditioners as above, grids over the whole
    range (``_side``), loads and moduli as in practice."""
    kind = rng.choice(["apply"] * 8 + ["build", "tangential", "solve", "nested", "adjoint",
                                       "ensemble"])
    backend = rng.choice(["fft", "periodic"])
    pn = math.exp(rng.uniform(math.log(0.002), math.log(0.02)))
    case = _drawn(rng, kind, backend, pn)
    case["E"] = round(rng.uniform(0.2, 5.0), 3)
    return case


def _drawn(rng, kind, backend, pn):
    if kind == "apply":
        return dict(kind=kind, backend=backend, Ns=_side(rng, 20, 4096),
                    bits=rng.choice([32, 64]))
    if kind == "build":
        return dict(kind=kind, backend="fft", Ns=_side(rng, 32, 1500), bits=rng.choice([32, 64]))
    if kind == "tangential":
        return dict(kind=kind, Ns=1 << rng.randint(5, 11), bits=rng.choice([32, 64]))
    if kind == "solve":
        return dict(kind=kind, backend=backend, Ns=_side(rng, 64, 400),
                    precond=rng.choice(["fourier", "fourier-fft"]), p_nominal=pn)
    if kind == "nested":
        return dict(kind=kind, backend=backend, Ns=64 * (1 << rng.randint(1, 4)),
                    engine=rng.choice(["auto", "fft"]),
                    active=backend == "fft" and rng.random() < 0.5, p_nominal=pn)
    if kind == "adjoint":
        return dict(kind=kind, backend=backend, Ns=_side(rng, 64, 512), p_nominal=pn)
    return dict(kind=kind, count=rng.randint(3, 8), smallest=64 << rng.randint(0, 1),
                largest=256, p_nominal=pn)


# ── inputs ────────────────────────────────────────────────────────────────────

def _generator(seed):
    return torch.Generator().manual_seed(1000003 * int(seed) + 17)


def _pressure(Ns, seed, parts=1):
    """Pressures of a partial contact: zero on most of the grid."""
    p = torch.randn(parts * Ns * Ns, generator=_generator(seed), dtype=torch.float64)
    return (p - 0.8).clamp_(min=0.0)


def _rough_gap(Ns, seed, H=0.8, k_low=4.0, k_high=64.0, rms=0.002):
    """Gap of a self-affine rough surface (random phases, power-law
    amplitudes between two wavenumbers), flat, C-contiguous float64."""
    k = np.fft.fftfreq(Ns, 1.0 / Ns)
    m = np.hypot(k[:, None], k[None, :])
    m[0, 0] = 1.0
    amp = np.where((m >= k_low) & (m <= k_high), m ** (-1.0 - H), 0.0)
    phase = torch.rand(Ns, Ns, generator=_generator(seed), dtype=torch.float64).numpy()
    h = np.fft.ifft2(amp * np.exp(2j * np.pi * phase)).real
    h -= h.mean()
    return np.ascontiguousarray(-(h * (rms / h.std()))).ravel()


def _members(case):
    """Sides and backends of an ensemble: sides between the two given."""
    sides = []
    n = case["smallest"]
    while n <= case["largest"]:
        sides.append(n)
        n *= 2
    return [(sides[i % len(sides)], "fft" if i % 2 else "periodic")
            for i in range(case["count"])]


def _modulus(case):
    return case.get("E", 1.0)


def _solver(case):
    return api.ContactSolver(case["Ns"], E_star=_modulus(case), backend=case["backend"])


def _dtype(case):
    return torch.float64 if case["bits"] == 64 else torch.float32


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("apply", "build"):
        s["x"] = _pressure(case["Ns"], seed).to(_dtype(case)).cuda()
        s["y"] = torch.empty_like(s["x"])
        if kind == "apply":
            s["solver"] = _solver(case)
    elif kind == "tangential":
        s["x"] = torch.randn(2 * case["Ns"] ** 2, generator=_generator(seed),
                             dtype=torch.float64).to(_dtype(case)).cuda()
        s["y"] = torch.empty_like(s["x"])
        s["solver"] = TangentialFFTOperator(case["Ns"], 1.0, _modulus(case), 0.3)
    elif kind == "solve":
        s["gap"] = _rough_gap(case["Ns"], seed)
        s["solver"] = _solver(case)
    elif kind == "nested":
        s["gap"] = torch.from_numpy(_rough_gap(case["Ns"], seed)).cuda()
    elif kind == "adjoint":
        Ns = case["Ns"]
        s["solver"] = _solver(case)
        s["result"] = s["solver"].solve(_rough_gap(Ns, seed), case["p_nominal"], tol=SOLVE_TOL,
                                        precond="fourier-fft")
        s["w"] = _weights(Ns, seed).cuda()
        s["grad"] = torch.empty_like(s["w"])
    else:
        s["gaps"] = [torch.from_numpy(_rough_gap(n, 100 * seed + i, k_high=min(64.0, n / 4)))
                     .cuda() for i, (n, _) in enumerate(_members(case))]
        s["problems"] = [dict(backend=b, grid_size=n, p_nominal=case["p_nominal"],
                              E_star=_modulus(case), gap_ptr=g.data_ptr())
                         for g, (n, b) in zip(s["gaps"], _members(case))]
    torch.cuda.synchronize()
    return s


def _weights(Ns, seed):
    """dL/dp of a smooth loss."""
    x = torch.arange(Ns, dtype=torch.float64) / Ns
    a = torch.rand(4, generator=_generator(seed + 7), dtype=torch.float64) * 2 * math.pi
    return (torch.sin(2 * math.pi * x + a[0])[:, None] * torch.cos(4 * math.pi * x + a[1])[None, :]
            + torch.cos(6 * math.pi * x + a[2])[None, :] * 0.5 + 1.0).reshape(-1).contiguous()


def _fields(r):
    return dict(pressure=r.pressure, displacement=r.displacement, gap=r.gap,
                objective=r.objective, approach=r.approach)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("apply", "tangential"):
        state["solver"].matvec_device(state["x"].data_ptr(), state["y"].data_ptr(),
                                      case["bits"])
        return state["y"]
    if kind == "build":
        solver = _solver(case)
        solver.matvec_device(state["x"].data_ptr(), state["y"].data_ptr(), case["bits"])
        return state["y"]
    if kind == "solve":
        return _fields(state["solver"].solve(state["gap"], case["p_nominal"], tol=SOLVE_TOL,
                                             precond=case["precond"]))
    if kind == "nested":
        return _fields(api.solve_nested_device(
            case["Ns"], state["gap"].data_ptr(), case["p_nominal"], tol=SOLVE_TOL,
            E_star=_modulus(case), backend=case["backend"], precision="double",
            precond_engine=case["engine"], active_set=case["active"], reuse_operators=True))
    if kind == "adjoint":
        g, _ = state["solver"].adjoint_device(state["result"], state["w"].data_ptr(),
                                              state["grad"].data_ptr(), tol=SOLVE_TOL)
        return dict(grad_gap=state["grad"], grad_p_nominal=g)
    results, _ = api.solve_ensemble_device(state["problems"], tol=SOLVE_TOL, precision="double")
    return [_fields(r) for r in results]


# ── what a pass cannot do without ─────────────────────────────────────────────

def _apply_work(backend, Ns, real_bytes, components=1, tables=1):
    """Input and output once, the kernel spectrum once (free space), and the
    operations of a real 2-D transform pair. A response on one chip also
    needs its half spectrum stored and read twice where it exceeds a
    workgroup's memory; that is the method's, not counted here."""
    n = 2 * Ns if backend == "fft" else Ns
    nbytes = components * 2 * Ns * Ns * real_bytes
    if backend == "fft":
        nbytes += tables * (Ns + 1) ** 2 * real_bytes
    # rows and columns that are not all zero, 2.5 n log2 n each, both ways
    rows = components * 2 * Ns * 2.5 * n * math.log2(n)
    cols = components * 2 * (n // 2 + 1) * 5.0 * n * math.log2(n)
    return nbytes, rows + cols


def work(case):
    kind = case["kind"]
    b = case.get("bits", 64) // 8
    if kind in ("apply", "build"):
        nbytes, flops = _apply_work(case["backend"], case["Ns"], b)
        if kind == "build":   # the influence table and its transform
            nbytes += (case["Ns"] + 1) ** 2 * 8
            flops *= 2
    elif kind == "tangential":
        nbytes, flops = _apply_work("fft", case["Ns"], b, components=2, tables=3)
    else:
        # iterations a preconditioned solve of these surfaces needs at least,
        # two responses and one preconditioner each (adjoint: one and one)
        sides = ([(case["Ns"], case["backend"])] if kind != "ensemble" else _members(case))
        its, applies = (30, 1) if kind == "adjoint" else (40, 2)
        nbytes = flops = 0.0
        for Ns, backend in sides:
            ab, af = _apply_work(backend, Ns, 8)
            pb, pf = _apply_work("periodic", Ns, 8)
            nbytes += its * (applies * ab + pb)
            flops += its * (applies * af + pf)
    return {"bytes": float(nbytes), "flops": float(flops)}


# ── the same results in 64 bits, without the library ─────────────────────────

def _log_ratio(t, s1, s2):
    """t log((s1 + |(t, s1)|)/(s2 + |(t, s2)|)), stable for s1 near s2."""
    r1, r2 = torch.sqrt(t * t + s1 * s1), torch.sqrt(t * t + s2 * s2)
    return t * torch.log1p(((s1 - s2) + (s1 - s2) * (s1 + s2) / (r1 + r2)) / (s2 + r2))


def _offsets(Ns):
    d = torch.arange(Ns, dtype=torch.float64)
    return d[None, :], d[:, None]


def _love_unit(x, y):
    """Potential of a uniform unit square at offset (x, y) >= 0 from its
    centre: integral of 1/r (Love 1929)."""
    xp, xm, yp, ym = x + 0.5, x - 0.5, y + 0.5, y - 0.5
    return (_log_ratio(xp, yp, ym) - _log_ratio(xm, yp, ym)
            + _log_ratio(yp, xp, xm) - _log_ratio(ym, xp, xm))


def _spectrum(table, odd=False):
    """Transform of a table of offsets 0 .. Ns-1, continued evenly (or oddly
    in both axes) to negative offsets on a torus of side 2 Ns."""
    Ns = table.shape[0]
    full = torch.zeros(2 * Ns, 2 * Ns, dtype=torch.float64)
    sgn = -1.0 if odd else 1.0
    full[:Ns, :Ns] = table
    full[Ns + 1:, :Ns] = sgn * table[1:].flip(0)
    full[:Ns, Ns + 1:] = sgn * table[:, 1:].flip(1)
    full[Ns + 1:, Ns + 1:] = table[1:, 1:].flip(0).flip(1)
    if odd:
        full[0, :] = 0.0
        full[:, 0] = 0.0
    return torch.fft.rfft2(full)


class _Response:
    """u = S p of a unit domain in 64 bits."""

    def __init__(self, backend, Ns, E):
        self.Ns = Ns
        if backend == "fft":
            self.n = 2 * Ns
            self.K = _spectrum(_love_unit(*_offsets(Ns)) / (Ns * math.pi * E))
        else:
            self.n = Ns
            k = torch.fft.fftfreq(Ns, 1.0 / Ns, dtype=torch.float64)
            q = 2 * math.pi * torch.hypot(k[:, None], k[None, : Ns // 2 + 1].abs())
            q[0, 0] = 1.0
            self.K = 2.0 / (q * E)
            self.K[0, 0] = 0.0

    def __call__(self, p):
        n, Ns = self.n, self.Ns
        return torch.fft.irfft2(torch.fft.rfft2(p, s=(n, n)) * self.K, s=(n, n))[:Ns, :Ns]


def _tangential_exact(Ns, q, E, nu=0.3):
    """Shear tractions on unit squares (Cerruti), 2x2 block convolution."""
    x, y = _offsets(Ns)
    xp, xm, yp, ym = x + 0.5, x - 0.5, y + 0.5, y - 0.5
    along = _log_ratio(yp, xp, xm) - _log_ratio(ym, xp, xm)
    xx = (1 - nu) * _love_unit(x, y) + nu * along
    rpp, rpm = torch.hypot(xp, yp), torch.hypot(xp, ym)
    rmp, rmm = torch.hypot(xm, yp), torch.hypot(xm, ym)
    xy = nu * 2.0 * y * (1.0 / (rmp + rmm) - 1.0 / (rpp + rpm))
    f = 1.0 / (Ns * math.pi * E * (1 - nu))
    Kxx, Kyy, Kxy = _spectrum(f * xx), _spectrum(f * xx.T), _spectrum(f * xy, odd=True)
    n = 2 * Ns
    a = torch.fft.rfft2(q[:Ns * Ns].reshape(Ns, Ns), s=(n, n))
    b = torch.fft.rfft2(q[Ns * Ns:].reshape(Ns, Ns), s=(n, n))
    u = torch.fft.irfft2(Kxx * a + Kxy * b, s=(n, n))[:Ns, :Ns]
    v = torch.fft.irfft2(Kxy * a + Kyy * b, s=(n, n))[:Ns, :Ns]
    return torch.cat([u.reshape(-1), v.reshape(-1)])


def _on_support(S, C, rhs, x0, steps=2000, rel=1e-15):
    """Solve S x = rhs - const on the points C with sum x = sum x0, x = 0
    elsewhere: conjugate gradients in the zero-sum subspace."""
    nc = float(C.sum())
    cut = lambda v: torch.where(C, v - v[C].sum() / nc, 0.0)   # noqa: E731
    x = x0.clone()
    r = cut(rhs - S(x))
    d, rr, first = r.clone(), float((r * r).sum()), None
    for _ in range(steps):
        first = rr if first is None else first
        if rr <= rel * rel * first or rr == 0.0:
            break
        q = cut(S(d))
        a = rr / float((d * q).sum())
        x += a * d
        r -= a * q
        rr, old = float((r * r).sum()), rr
        d = r + (rr / old) * d
    return x


def _contact(S, gap, p_nominal):
    """The pressure p >= 0 of mean p_nominal that minimises p.S p/2 + gap.p,
    by changing the support until no pressure is negative and no point
    outside it lies below the contact plane."""
    N = gap.numel()
    C = gap < torch.quantile(gap.reshape(-1)[:: max(1, N // 100000)], 0.3)
    p = torch.where(C, p_nominal * N / float(C.sum()), 0.0)
    for outer in range(60):
        last = outer >= 12
        p = _on_support(S, C, -gap, p, steps=2000 if last else 40,
                        rel=1e-14 if last else 1e-3)
        keep = C & (p > 0)
        g = S(p) + gap
        touch = ~C & (g < g[C].mean())
        p = torch.where(keep, p, 0.0)
        p *= p_nominal * N / float(p.sum())
        same = bool((keep == C).all()) and not bool(touch.any())
        C = keep | touch
        if same and last:
            return p, C
    return None, None


def exact(case, seed):
    kind = case["kind"]
    if kind in ("apply", "build"):
        Ns = case["Ns"]
        p = _pressure(Ns, seed).to(_dtype(case)).double().reshape(Ns, Ns)
        return _Response(case["backend"], Ns, _modulus(case))(p).reshape(-1)
    if kind == "tangential":
        q = torch.randn(2 * case["Ns"] ** 2, generator=_generator(seed), dtype=torch.float64)
        return _tangential_exact(case["Ns"], q.to(_dtype(case)).double(),
                                 _modulus(case))
    # solves of larger grids, nested ones and ensembles take minutes on a host
    if kind not in ("solve", "adjoint") or case["Ns"] > (
            300 if case["backend"] == "fft" else 512):
        return None
    Ns = case["Ns"]
    S = _Response(case["backend"], Ns, _modulus(case))
    gap = torch.from_numpy(_rough_gap(Ns, seed)).reshape(Ns, Ns)
    p, C = _contact(S, gap, case["p_nominal"])
    if p is None:
        return None
    if kind == "solve":
        u = S(p)
        g = u + gap
        plane = float(g[C].mean())
        return dict(pressure=p, displacement=u, gap=None,
                    objective=float((p * (0.5 * u + gap)).sum()), approach=plane)
    w = _weights(Ns, seed).reshape(Ns, Ns)
    mu = _on_support(S, C, w, torch.zeros_like(w))
    nu = float((w - S(mu))[C].mean())
    return dict(grad_gap=-mu.reshape(-1), grad_p_nominal=nu * Ns * Ns)
