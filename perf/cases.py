"""Timing cases: the calls that programs built on this package spend their time in.

Each case is one call (or one burst of calls) through the public entry points:
the Python mirror's functions on host arrays, the `_d` entry points of the C
ABI on device buffers, and the request server.  `listed()` names the cases,
`draw()` gives more of the same ranges, `prepare()` makes what a program holds
before the call, `run()` makes the call, `work()` counts what the call cannot
do without, and `exact()` restates each result in plain torch, in 64 bits.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from __graft_entry__ import load_package

KINDS = ("TT", "TE", "M++", "M--")              # psx_mcm_kind 0..3
COV = ("TTTT", "EEEE", "TTTE", "TETE", "TEEE", "TEEE_PLANCK", "TTEE")   # psx_cov_kind 0..6
COV_ARITY = {"TTTT": (8, 4, 4), "EEEE": (8, 4, 4), "TTTE": (4, 4, 2), "TETE": (5, 4, 2),
             "TEEE": (4, 4, 2), "TEEE_PLANCK": (4, 4, 2), "TTEE": (2, 4, 0)}  # W, spectra, ratios
SERVED = ("TT", "TE", "PM", "TTTT", "EEEE", "TETE", "TTEE")
VP = ctypes.c_void_p


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # one block of a low-resolution (nside 32) analysis, host in and out: the
        # smallest call, all latency
        {"name": "mcm_tt_95", "op": "mcm", "spec": "TT", "lmin": 0, "lmax": 95},
        # the five blocks of a polarised analysis at nside 256, device resident
        {"name": "set_767", "op": "set", "lmin": 0, "lmax": 767},
        # the same at nside 1024: the benchmark's headline size
        {"name": "set_3071", "op": "set", "lmin": 0, "lmax": 3071},
        # the covariance block with the most W spectra, at the benchmark's lmax
        {"name": "cov_tttt_2508", "op": "cov", "kind": "TTTT", "lmin": 0, "lmax": 2508,
         "host": False},
        # a two-family covariance block of an nside-256 analysis from l = 2, host in and out
        {"name": "cov_tete_750", "op": "cov", "kind": "TETE", "lmin": 2, "lmax": 750,
         "host": True},
        # many mask cross-spectra against one family, on the matrix cores
        {"name": "batch_tt_64x1535", "op": "batch", "kind": "TT", "K": 64, "lmax": 1535,
         "precision": 1},
        # the mask -> W front end of four nside-1024 masks, host maps in
        {"name": "mask_spectra_4x1024", "op": "mask_spectra", "nside": 1024, "lmax": 3071,
         "nmaps": 4},
        # synthesis of one polarised sky, host a_lm in and host maps out
        {"name": "alm2map_pol_512", "op": "alm2map_pol", "nside": 512, "lmax": 1535},
        # the whole pipeline: two (I, Q, U) maps and four masks to nine spectra
        {"name": "master_512", "op": "master", "nside": 512, "lmin": 2},
        # decoupling one spectrum with the largest block of a TT analysis at lmax 6143
        {"name": "lu_solve_6144", "op": "lu", "n": 6144, "nrhs": 1},
        # decoupling a covariance block at the benchmark's lmax
        {"name": "decouple_2509", "op": "decouple", "n": 2509},
        # a burst of mixed requests to the server, results to the host
        {"name": "serve_24", "op": "serve", "requests": 24, "lo": 511, "hi": 1535},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["mcm", "set", "cov", "batch", "mask_spectra", "alm2map_pol", "master", "lu",
                     "decouple", "serve"])
    if op == "mcm":
        return {"op": op, "spec": rng.choice(KINDS), "lmin": rng.choice([0, 2]),
                "lmax": _log_int(rng, 60, 1535)}
    if op == "set":
        return {"op": op, "lmin": rng.choice([0, 2]), "lmax": _log_int(rng, 200, 3071)}
    if op == "cov":
        return {"op": op, "kind": rng.choice(COV), "lmin": rng.choice([0, 2]),
                "lmax": _log_int(rng, 200, 2508), "host": rng.random() < 0.5}
    if op == "batch":
        return {"op": op, "kind": rng.choice(KINDS), "K": rng.randint(8, 64),
                "lmax": _log_int(rng, 383, 1535), "precision": rng.choice([0, 1])}
    if op == "mask_spectra":
        nside = rng.choice([128, 256, 512, 1024])
        return {"op": op, "nside": nside, "lmax": rng.randint(2 * nside, 3 * nside - 1),
                "nmaps": rng.randint(1, 4)}
    if op == "alm2map_pol":
        nside = rng.choice([128, 256, 512])
        return {"op": op, "nside": nside, "lmax": rng.randint(2 * nside, 3 * nside - 1)}
    if op == "master":
        return {"op": op, "nside": rng.choice([64, 128, 256, 512]), "lmin": rng.randint(2, 20)}
    if op == "lu":
        return {"op": op, "n": _log_int(rng, 500, 6144), "nrhs": rng.randint(1, 4)}
    if op == "decouple":
        return {"op": op, "n": _log_int(rng, 250, 2509)}
    lo = rng.randint(200, 700)
    return {"op": op, "requests": rng.randint(6, 24), "lo": lo, "hi": rng.randint(lo, 1535)}


# ---- inputs ------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _mask_spectrum(rng, n, cross=False):
    """A spectrum of length n like an apodised cut-sky mask's: W_0 ~ 4 pi f_sky, a fall-off of
    ten decades with ripples; a cross-spectrum changes sign."""
    ell = np.arange(n, dtype=np.float64)
    W = 4 * np.pi * rng.uniform(0.45, 0.65) * np.exp(-ell / 40.0) * (1 + 0.2 * np.cos(ell / 7.0))
    W += 4 * np.pi * 1e-5 * np.exp(-ell / 600.0) * rng.uniform(0.5, 1.5, n)
    W += 4 * np.pi * 1e-9 * rng.uniform(0.0, 1.0, n)
    if cross:
        W *= np.where(rng.uniform(size=n) < 0.15, -0.3, 1.0)
    return W


def _signal_spectrum(rng, n):
    ell = np.arange(n, dtype=np.float64)
    return 1e3 * rng.uniform(0.5, 2.0) * (ell + 10.0) ** -2.5 * np.exp(-(ell / 2000.0) ** 2)


def _noise_ratio(rng, n):
    ell = np.arange(n, dtype=np.float64)
    return np.sqrt(1.0 + rng.uniform(0.0, 2.0) * (ell / n) ** 2)


def _cov_inputs(rng, kind, n):
    nW, nS, nR = COV_ARITY[kind]
    return ([_signal_spectrum(rng, n) for _ in range(nS)], [_noise_ratio(rng, n) for _ in range(nR)],
            [_mask_spectrum(rng, n) for _ in range(nW)])


def _set_inputs(rng, n):
    return [_mask_spectrum(rng, n, cross) for cross in (False, True, True, False)]


def _rings(nside):
    """(first pixel, pixel count, cos theta, phi0) of the 4 nside - 1 HEALPix rings."""
    i = np.arange(1, 4 * nside, dtype=np.int64)
    cap, south = i < nside, i > 3 * nside
    j = np.where(cap, i, np.where(south, 4 * nside - i, nside))
    count = 4 * j
    first = np.concatenate([[0], np.cumsum(count)[:-1]])
    z = np.where(cap, 1 - j * j / (3.0 * nside * nside),
                 np.where(south, -(1 - j * j / (3.0 * nside * nside)),
                          4.0 / 3.0 - 2.0 * i / (3.0 * nside)))
    shifted = cap | south | ((i - nside) % 2 == 0)
    return first, count, z, np.where(shifted, np.pi / count, 0.0)


def _directions(nside):
    first, count, z, phi0 = (torch.from_numpy(a).to(_device()) for a in _rings(nside))
    ring = torch.repeat_interleave(torch.arange(first.numel(), device=_device()), count)
    j = torch.arange(ring.numel(), device=_device()) - first[ring]
    return z[ring], phi0[ring] + 2 * math.pi * j / count[ring]


def _taper(x, width):
    t = torch.clamp(x / width, 0.0, 1.0)
    return 0.5 * (1.0 - torch.cos(math.pi * t))


def _masks(nside, count, seed, holes=40):
    """Galactic cut |b| < 20 degrees and random holes of 0.5 degrees, apodised over 1 degree."""
    z, phi = _directions(nside)
    rho = torch.sqrt((1 - z) * (1 + z))
    x, y = rho * torch.cos(phi), rho * torch.sin(phi)
    cut = _taper(torch.abs(torch.asin(z)) - math.radians(20.0), math.radians(1.0))
    rng = np.random.default_rng([seed, 1])
    out = []
    for _ in range(count):
        m = cut.clone()
        for _ in range(holes):
            v = rng.standard_normal(3)
            v /= np.linalg.norm(v)
            d = torch.acos(torch.clamp(x * v[0] + y * v[1] + z * v[2], -1.0, 1.0))
            m *= _taper(d - math.radians(0.5), math.radians(1.0))
        out.append(m)
    return torch.stack(out)


def _skies(nside, seed):
    """Two (I, Q, U) maps: a large-scale sky common to both and independent white noise."""
    z, phi = _directions(nside)
    g = _gen(seed)
    rng = np.random.default_rng([seed, 2])
    sky = torch.zeros(3, z.numel(), dtype=torch.float64, device=_device())
    for f, amp in enumerate((100.0, 10.0, 10.0)):
        for k in range(1, 9):
            a, b = rng.standard_normal(2)
            sky[f] += amp / k * (1 - z * z) * (a * torch.cos(k * phi) + b * torch.sin(k * phi) * z)
    return [sky + 5.0 * torch.randn(3, z.numel(), dtype=torch.float64, device=_device(),
                                    generator=g) for _ in range(2)]


def _coupling(n, g):
    """A matrix like a mode-coupling matrix: a narrow kernel about the diagonal with the
    (2 l2 + 1) / (2 l1 + 1) tilt and small random wings."""
    l = torch.arange(n, dtype=torch.float64, device=_device())
    d = torch.abs(l[:, None] - l[None, :])
    M = 0.6 * torch.exp(-d / 1.5) + 0.02 * torch.exp(-d / 60.0) * torch.rand(
        n, n, dtype=torch.float64, device=_device(), generator=g)
    return M * torch.sqrt((2 * l + 1)[None, :] / (2 * l + 1)[:, None])


def _covariance(n, g):
    l = torch.arange(n, dtype=torch.float64, device=_device())
    c = 1e3 * (l + 10.0) ** -2.5 + 1e-4
    d = torch.abs(l[:, None] - l[None, :])
    noise = torch.rand(n, n, dtype=torch.float64, device=_device(), generator=g)
    K = torch.exp(-d / 2.0) + 1e-3 * torch.exp(-d / 80.0) * (noise + noise.T)
    return torch.sqrt(c[:, None] * c[None, :]) * K


def _linear(case, seed):
    n, g = case["n"], _gen(seed)
    if case["op"] == "lu":
        A = _coupling(n, g)
        l = torch.arange(n, dtype=torch.float64, device=_device())[:, None]
        B = (l + 10.0) ** -2.0 * (1 + 0.1 * torch.randn(n, case["nrhs"], dtype=torch.float64,
                                                        device=_device(), generator=g))
        return A, B
    return _covariance(n, g), _coupling(n, g), _coupling(n, g)


def _alms(lmax, seed):
    """T, E, B coefficients of a Gaussian sky, (3, nalm), m-major."""
    g = _gen(seed)
    ls = torch.cat([torch.arange(m, lmax + 1, device=_device()) for m in range(lmax + 1)])
    a = torch.randn(3, ls.numel(), dtype=torch.complex128, device=_device(), generator=g)
    a[:, : lmax + 1] = a[:, : lmax + 1].real * math.sqrt(2.0) + 0j
    a[1:] *= (ls >= 2)
    amp = torch.tensor([1.0, 0.3, 0.1], dtype=torch.float64, device=_device())[:, None]
    return a * amp * (ls + 10.0) ** -1.25


def _requests(case):
    """The burst: (kind, lmax) of each request, lmax log-uniform in [lo, hi]."""
    rng = np.random.default_rng(17)
    sizes = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["requests"]))
    return [(SERVED[k % len(SERVED)], int(l))
            for k, l in zip(rng.permutation(case["requests"]), sizes)]


def _served_inputs(case, seed):
    """Resident spectra: 10 mask spectra (keys 0-9), 4 signal spectra (10-13), 4 noise ratios
    (14-17)."""
    rng, n = np.random.default_rng([seed, 4]), case["hi"] + 1
    return ([_mask_spectrum(rng, n) for _ in range(10)] + [_signal_spectrum(rng, n) for _ in range(4)]
            + [_noise_ratio(rng, n) for _ in range(4)])


def _host(t):
    return t.cpu().numpy()


def _fortran(t):
    return np.asfortranarray(t.T.contiguous().cpu().numpy().T)


def prepare(case, seed):
    pkg, op = load_package(), case["op"]
    ctx = pkg.default_context()
    rng = np.random.default_rng([seed, 0])
    s = {"case": case, "pkg": pkg, "ctx": ctx}
    dev = lambda a: torch.from_numpy(a).to(_device())  # noqa: E731
    if op == "mcm":
        s["W"] = _mask_spectrum(rng, case["lmax"] + 1, case["spec"] == "TE")
    elif op == "set":
        n = case["lmax"] - case["lmin"] + 1
        s["W"] = [dev(w) for w in _set_inputs(rng, case["lmax"] + 1)]
        s["out"] = [torch.empty(n, n, dtype=torch.float64, device=_device()) for _ in range(5)]
    elif op == "cov":
        s["in"] = _cov_inputs(rng, case["kind"], case["lmax"] + 1)
        if not case["host"]:
            n = case["lmax"] - case["lmin"] + 1
            s["in"] = tuple([dev(a) for a in group] for group in s["in"])
            s["ptr"] = tuple((VP * 8)(*[VP(t.data_ptr()) for t in group]) for group in s["in"])
            s["out"] = torch.empty(n, n, dtype=torch.float64, device=_device())
    elif op == "batch":
        n = case["lmax"] + 1
        s["W"] = [dev(_mask_spectrum(rng, n)) for _ in range(case["K"])]
        s["out"] = torch.empty(case["K"], n, n, dtype=torch.float64, device=_device())
        s["Wp"] = (VP * case["K"])(*[VP(w.data_ptr()) for w in s["W"]])
        s["outp"] = (VP * case["K"])(*[VP(o.data_ptr()) for o in s["out"]])
    elif op == "mask_spectra":
        s["maps"] = _host(_masks(case["nside"], case["nmaps"], seed))
    elif op == "alm2map_pol":
        s["alms"] = _host(_alms(case["lmax"], seed))
    elif op == "master":
        s["maps"] = [list(_host(m)) for m in _skies(case["nside"], seed)]
        s["masks"] = list(_host(_masks(case["nside"], 4, seed)))
    elif op == "lu":
        A, B = _linear(case, seed)
        s["A"], s["B"] = _fortran(A), _fortran(B)
    elif op == "decouple":
        s["Y"], s["B1"], s["B2"] = (_fortran(t) for t in _linear(case, seed))
    elif op == "serve":
        s["srv"] = srv = pkg.Server(ctx, slots=4, arena_bytes=1 << 30, lmax_max=case["hi"])
        for k, v in enumerate(_served_inputs(case, seed)):
            srv.put(k, v)
        s["rq"] = []
        for kind, lmax in _requests(case):
            n = lmax + 1
            s["rq"].append((kind, lmax, [np.empty((n, n), order="F")
                                         for _ in range(2 if kind == "PM" else 1)]))
    return s


# ---- the calls ---------------------------------------------------------------
def run(s):
    case, ctx, pkg = s["case"], s["ctx"], s["pkg"]
    op, L = case["op"], ctx.lib
    if op == "mcm":
        return pkg.mcm_from_spectrum(case["spec"], s["W"], lmin=case["lmin"], lmax=case["lmax"],
                                     ctx=ctx).parent
    if op == "set":
        lmin, lmax = case["lmin"], case["lmax"]
        ctx.check(L.psx_mcm_set_d(ctx.handle, lmin, lmax, lmax + 1, *[w.data_ptr() for w in s["W"]],
                                  *[o.data_ptr() for o in s["out"]], lmax - lmin + 1),
                  "psx_mcm_set_d")
        return s["out"]
    if op == "cov":
        lmin, lmax, kind = case["lmin"], case["lmax"], COV.index(case["kind"])
        if case["host"]:
            return ctx.cov(kind, lmin, lmax, *s["in"])
        sp, rp, wp = s["ptr"]
        ctx.check(L.psx_cov_d(ctx.handle, kind, lmin, lmax, sp, rp, wp, lmax + 1, 0,
                              s["out"].data_ptr(), lmax - lmin + 1), "psx_cov_d")
        return s["out"]
    if op == "batch":
        n = case["lmax"] + 1
        ctx.check(L.psx_mcm_batch_d(ctx.handle, KINDS.index(case["kind"]), 0, case["lmax"],
                                    case["K"], s["Wp"], n, case["precision"], s["outp"], n),
                  "psx_mcm_batch_d")
        return s["out"]
    if op == "mask_spectra":
        return ctx.mask_spectra(s["maps"], case["nside"], case["lmax"], 3)
    if op == "alm2map_pol":
        return ctx.alm2map_pol(s["alms"], case["nside"], case["lmax"])
    if op == "master":
        (T1, P1, T2, P2), (m1, m2) = s["masks"], s["maps"]
        out = pkg.master(m1, T1, P1, m2, T2, P2, lmin=case["lmin"], ctx=ctx)
        return {k: v.parent for k, v in out.items()}
    if op == "lu":
        return ctx.lu_solve(s["A"], s["B"])
    if op == "decouple":
        return ctx.decouple_covmat(s["Y"], s["B1"], s["B2"])
    srv, tickets = s["srv"], []
    for i, (kind, lmax, out) in enumerate(s["rq"]):
        W = [(i + k) % 10 for k in range(8)]
        if kind == "PM":
            t = srv.submit(1, lmax=lmax, W=W[:1], out=out)
        elif kind in KINDS:
            t = srv.submit(0, kind=KINDS.index(kind), lmax=lmax, W=W[:1], out=out)
        else:
            nW, nS, nR = COV_ARITY[kind]
            t = srv.submit(3, kind=COV.index(kind), lmax=lmax, W=W[:nW],
                           spectra=range(10, 10 + nS), ratios=range(14, 14 + nR), out=out)
        tickets.append(t)
    for t in tickets:
        srv.wait(t)
        srv.release(t)
    return [out for _, _, out in s["rq"]]


# ---- what a call cannot do without -------------------------------------------
def _terms(lmin, lmax, LW):
    """(l1 <= l2, l3) terms with even l1 + l2 + l3 and l3 < LW."""
    total = 0
    for l1 in range(lmin, lmax + 1):
        S = l1 + np.arange(l1, lmax + 1, dtype=np.int64)
        total += int(np.maximum(0, l1 - np.maximum(0, (S - LW + 2) // 2) + 1).sum())
    return total


# flops of one term in closed form: the family product and its polynomial, and one multiply-add
# for each W spectrum
_MCM_FLOPS = {"TT": 3, "TE": 7, "M++": 8, "M--": 7, "PM": 15}


def _cov_flops(kind):
    base = {"TTTT": 1, "EEEE": 6, "TTTE": 1, "TETE": 5, "TEEE": 5, "TEEE_PLANCK": 6, "TTEE": 1}
    return base[kind] + 2 * COV_ARITY[kind][0]


def _transform_flops(nside, lmax, spin0, spin2, passes):
    """Ring sums of `passes` transforms of spin0 scalar and spin2 polarised fields over the
    2 nside ring pairs: the recurrences once for all, multiply-adds for each field."""
    steps = (lmax + 1) * (lmax + 2) // 2 * 2 * nside
    return passes * steps * ((4 + 4 * spin0 if spin0 else 0) + (9 + 16 * spin2 if spin2 else 0))


def work(case):
    op = case["op"]
    if op in ("mcm", "set", "cov"):
        lmin, lmax = case["lmin"], case["lmax"]
        n, t = lmax - lmin + 1, _terms(lmin, lmax, lmax + 1)
        if op == "mcm":
            return {"bytes": 8 * (lmax + 1 + n * n), "flops": _MCM_FLOPS[case["spec"]] * t}
        if op == "set":
            return {"bytes": 8 * (4 * (lmax + 1) + 5 * n * n), "flops": 20 * t}
        return {"bytes": 8 * (sum(COV_ARITY[case["kind"]]) * (lmax + 1) + n * n),
                "flops": _cov_flops(case["kind"]) * t}
    if op == "batch":
        n, K = case["lmax"] + 1, case["K"]
        return {"bytes": 8 * K * (n + n * n),
                "flops": (_MCM_FLOPS[case["kind"]] + 2 * (K - 1)) * _terms(0, n - 1, n)}
    if op in ("mask_spectra", "alm2map_pol", "master"):
        nside = case["nside"]
        npix, lmax = 12 * nside * nside, case.get("lmax", 3 * nside - 1)
        if op == "mask_spectra":
            m = case["nmaps"]
            return {"bytes": 8 * (m * npix + m * m * (lmax + 1)),
                    "flops": _transform_flops(nside, lmax, m, 0, 7)}
        if op == "alm2map_pol":
            return {"bytes": 8 * 3 * npix + 16 * 3 * (lmax + 1) * (lmax + 2) // 2,
                    "flops": _transform_flops(nside, lmax, 1, 1, 1)}
        n = lmax - case["lmin"] + 1
        return {"bytes": 8 * (10 * npix + 9 * n),
                "flops": _transform_flops(nside, lmax, 6, 2, 7) + 20 * _terms(0, lmax, lmax + 1)
                + 2 * n ** 3 // 3 * (3 + 8)}
    if op == "lu":
        n, r = case["n"], case["nrhs"]
        return {"bytes": 8 * (n * n + 2 * n * r), "flops": 2 * n ** 3 // 3 + 2 * n * n * r}
    if op == "decouple":
        n = case["n"]
        return {"bytes": 8 * 4 * n * n, "flops": 2 * (2 * n ** 3 // 3) + 4 * n ** 3}
    total = {"bytes": 0, "flops": 0}
    for kind, lmax in _requests(case):
        n, t = lmax + 1, _terms(0, lmax, lmax + 1)
        total["bytes"] += 8 * n * n * (2 if kind == "PM" else 1)
        total["flops"] += t * (_MCM_FLOPS[kind] if kind in _MCM_FLOPS else _cov_flops(kind))
    return total


# ---- the results in plain torch, 64 bits --------------------------------------
def _projectors(lmin, lmax, families):
    """Sums over l3 of What(l3) times the 3j product of each family, for l1, l2 = lmin..lmax.

    families: (name, [W, ...]) with name one of TT, TE, M++, M--; the products in closed form
    from gamma_m = C(2m, m) / 4^m.  Returns one list of matrices a family."""
    dev, n = _device(), lmax + 1
    m = np.arange(1, 4 * n + 8, dtype=np.longdouble)
    g = np.concatenate([[np.longdouble(1)], np.cumprod((2 * m - 1) / (2 * m))])
    k = np.arange(g.size, dtype=np.longdouble)
    tab = lambda a: torch.from_numpy(a.astype(np.float64)).to(dev)  # noqa: E731
    G, Z, D, IG = tab(g), tab((2 * k + 1) * g), tab(1 / ((2 * k + 1) * g)), tab(1 / g)
    ell = torch.arange(n, dtype=torch.float64, device=dev)
    P = ell * (ell + 1)
    sigma, prod = P[:, None] + P[None, :] - 1.0, P[:, None] * P[None, :]
    hat, out = [], []
    for _, Ws in families:
        h = []
        for W in Ws:
            w = torch.zeros(2 * n + 4, dtype=torch.float64, device=dev)
            w[: min(n, len(W))] = torch.as_tensor(np.asarray(W)[:n], device=dev)
            h.append(w * (2 * torch.arange(w.numel(), device=dev) + 1) / (4 * math.pi))
        hat.append(h)
        out.append([torch.zeros(n, n, dtype=torch.float64, device=dev) for _ in Ws])
    T = torch.arange(2 * n + 4, dtype=torch.float64, device=dev)
    T = T * (T + 1)
    hankel = lambda v, r: v[: 2 * r - 1].as_strided((r, r), (1, 1))  # noqa: E731
    for c in range(n):
        r = n - c                                  # l1, l2 = c .. lmax; l3 = l1 + l2 - 2c
        even = torch.outer(G[:r], G[:r]) * hankel(G[c] * D[c: c + 2 * r], r)
        Q = odd = None
        for (name, Ws), h, o in zip(families, hat, out):
            if name == "M--":
                if r < 2:
                    continue
                q = r - 1                          # l1, l2 = c+1 .. lmax; l3 = l1 + l2 - 2c - 1
                odd = torch.outer(Z[:q], Z[:q]) * hankel(Z[c] * IG[c + 2: c + 2 + 2 * q], q)
                d1 = sigma[c + 1:, c + 1:] - 1.0 - hankel(T[1: 1 + 2 * q], q)
                t = odd * d1 * d1
                for w, x in zip(h, o):
                    x[c + 1:, c + 1:] += t * hankel(w[1: 1 + 2 * q], q)
                continue
            t = even
            if name != "TT":
                if Q is None:
                    E = sigma[c:, c:] - hankel(T[: 2 * r], r)
                    Q = E * E - 1.0 - 2.0 * prod[c:, c:]
                t = even * Q if name == "TE" else even * Q * Q
            for w, x in zip(h, o):
                x[c:, c:] += t * hankel(w[: 2 * r], r)
    pi = (ell - 1) * ell * (ell + 1) * (ell + 2)
    pi = pi[:, None] * pi[None, :]
    inv = torch.where(pi > 0, 1.0 / torch.where(pi > 0, pi, torch.ones_like(pi)),
                      torch.zeros_like(pi))
    inv[:2] = 0
    inv[:, :2] = 0
    for (name, _), o in zip(families, out):
        for i, x in enumerate(o):
            if name == "TE":
                x = x * torch.sqrt(inv) / 2
            elif name != "TT":
                x = x * inv / 4
            o[i] = x[lmin:, lmin:]
    return out


def _blocks(lmin, lmax, families):
    ell = torch.arange(lmin, lmax + 1, dtype=torch.float64, device=_device())
    return [[(2 * ell + 1)[None, :] * x for x in o] for o in _projectors(lmin, lmax, families)]


def _cov_exact(kind, lmin, lmax, S, R, W):
    if kind == "TETE":
        te, tt = _projectors(lmin, lmax, [("TE", [W[0], W[2], W[3], W[4]]), ("TT", [W[1]])])
        x = [te[0], tt[0], te[1], te[2], te[3]]
    else:
        family = {"EEEE": "M++", "TEEE": "TE", "TEEE_PLANCK": "M++"}.get(kind, "TT")
        x = _projectors(lmin, lmax, [(family, W)])[0]
    n = lmax + 1
    vec = lambda a: torch.as_tensor(np.asarray(a)[lmin:n], device=_device())  # noqa: E731
    S, R = [vec(a) for a in S], [vec(a) for a in R]
    both = lambda *v: math.prod([a[:, None] * a[None, :] for a in v])  # noqa: E731
    plus = lambda a: a[:, None] + a[None, :]  # noqa: E731
    sq = torch.sqrt
    if kind in ("TTTT", "EEEE"):
        ip, jq, iq, jp = S
        rip, rjq, riq, rjp = R
        return (sq(both(ip, jq)) * x[0] + sq(both(iq, jp)) * x[1] + sq(both(ip)) * both(rjq) * x[2]
                + sq(both(jq)) * both(rip) * x[3] + sq(both(iq)) * both(rjp) * x[4]
                + sq(both(jp)) * both(riq) * x[5] + both(rip, rjq) * x[6] + both(riq, rjp) * x[7])
    if kind == "TTTE":
        ip, jp, iq, jq = S
        return (sq(both(ip)) * plus(jq) * x[0] + sq(both(jp)) * plus(iq) * x[1]
                + plus(jq) * both(R[0]) * x[2] + plus(iq) * both(R[1]) * x[3]) / 2
    if kind == "TETE":
        ip, jq, iq, jp = S
        cross = iq[:, None] * jp[None, :] + jp[:, None] * iq[None, :]
        return (sq(both(ip, jq)) * x[0] + 0.5 * cross * x[1] + sq(both(ip)) * both(R[1]) * x[2]
                + sq(both(jq)) * both(R[0]) * x[3] + both(R[0], R[1]) * x[4])
    if kind in ("TEEE", "TEEE_PLANCK"):
        jq, jp, ip, iq = S
        return (sq(both(jq)) * plus(ip) * x[0] + sq(both(jp)) * plus(iq) * x[1]
                + plus(ip) * both(R[0]) * x[2] + plus(iq) * both(R[1]) * x[3]) / 2
    ip, iq, jq, jp = S
    a = ip[:, None] * jq[None, :] + jq[:, None] * ip[None, :]
    b = iq[:, None] * jp[None, :] + jp[:, None] * iq[None, :]
    return (a * x[0] + b * x[1]) / 2


class _Sphere:
    """Spherical-harmonic sums on the HEALPix rings, one l at a time for every m and ring.

    The harmonics N_l d^l_{m,p}(theta) follow the three-term recurrence in l from their value at
    l = max(m, |p|), carried as mantissa x 2^(512 s) since they underflow near the poles."""

    def __init__(self, nside, lmax):
        self.nside, self.lmax, self.npix = nside, lmax, 12 * nside * nside
        self.first, self.count, z, phi0 = _rings(nside)
        dev = _device()
        self.z = torch.from_numpy(z).to(dev)
        self.ms = torch.arange(lmax + 1, dtype=torch.float64, device=dev)
        ld = np.longdouble
        j = np.minimum(np.arange(1, 4 * nside), 4 * nside - np.arange(1, 4 * nside)).astype(ld)
        i = np.arange(1, 4 * nside).astype(ld)
        cap = j < nside
        up = z > 0
        # 1 - |z| without cancellation, then 1 - z and 1 + z
        near = np.where(cap, j * j / (3 * ld(nside) ** 2),
                        1 - np.abs(ld(4) / 3 - 2 * i / (3 * ld(nside))))
        far = 2 - near
        minus, plus = np.where(up, near, far), np.where(up, far, near)
        self.log_c, self.log_s = np.log2(plus / 2) / 2, np.log2(minus / 2) / 2  # cos, sin theta/2
        self.lg = np.concatenate([[ld(0)], np.cumsum(np.log2(np.arange(1, 2 * lmax + 9, dtype=ld)))])
        self._starts = {}
        self.phase = torch.exp(-1j * self.ms[:, None] * torch.from_numpy(phi0).to(dev)[None, :])

    def starts(self, p):
        """(mantissa, scale) of d^l_{m,p} at l = max(m, |p|) for every m and ring."""
        if p in self._starts:
            return tuple(t.clone() for t in self._starts[p])
        m = np.arange(self.lmax + 1)
        lead = np.maximum(m, abs(p))
        # d^j_{j,b} = (-1)^(j-b) sqrt((2j)! / ((j+b)! (j-b)!)) cos^(j+b) sin^(j-b), moved to
        # m < |p| by d_{m,p} = (-1)^(m-p) d_{p,m} and d_{m,-p} = d_{p,-m}
        b = np.where(m >= abs(p), p, m if p >= 0 else -m)
        sign = (-1.0) ** (lead - b) * np.where((m < abs(p)) & (p > 0), (-1.0) ** (m - p), 1.0)
        coef = (self.lg[2 * lead] - self.lg[lead + b] - self.lg[lead - b]) / 2
        v = (coef[:, None] + (lead + b)[:, None] * self.log_c[None, :]
             + (lead - b)[:, None] * self.log_s[None, :])
        s = np.minimum(np.ceil(v / 512), 0)
        man = sign[:, None] * np.exp2((v - 512 * s).astype(np.float64))
        self._starts[p] = (torch.from_numpy(man).to(_device()),
                           torch.from_numpy(s.astype(np.int16)).to(_device()))
        return self.starts(p)

    def rows(self, spins):
        """Yields (l, [harmonics of rows m = 0..min(l, lmax) for each spin index p])."""
        L, state = self.lmax, []
        for p in spins:
            man, s = self.starts(p)
            state.append([p, torch.zeros_like(man), man, s])
        mm = self.ms
        for l in range(L + 1):
            vals = []
            for st in state:
                p, prev, cur, s = st
                if l < abs(p):
                    vals.append(None)
                    continue
                top = l + 1
                if l > abs(p):
                    # rows m < l step from l - 1; row l starts here
                    k, old = l - 1, l
                    m = mm[:old]
                    den = k * torch.sqrt((l * l - m * m) * (l * l - p * p)) if k else None
                    if k == 0:
                        nxt = self.z[None, :] * cur[:old]
                    else:
                        a = (2 * k + 1) / den
                        u = a[:, None] * (k * (k + 1) * self.z[None, :] - p * m[:, None])
                        w = l * torch.sqrt(torch.clamp((k * k - m * m) * (k * k - p * p), min=0)) / den
                        nxt = u * cur[:old] - w[:, None] * prev[:old]
                    prev[:old] = cur[:old]
                    cur[:old] = nxt
                    if l % 8 == 0:
                        big = torch.abs(cur[:old]) > 2.0 ** 256
                        big &= s[:old] < 0
                        f = torch.ones_like(cur[:old]).masked_fill_(big, 2.0 ** -512)
                        cur[:old] *= f
                        prev[:old] *= f
                        s[:old] += big.to(torch.int16)
                live = (s[:top] == 0).to(torch.float64)
                vals.append(cur[:top] * live * math.sqrt((2 * l + 1) / (4 * math.pi)))
            yield l, vals

    def _polar(self):
        """The rings of both caps: each has a length of its own, so they are transformed on the
        host (a GPU library would compile a plan for each)."""
        ns = self.nside
        return [(k, int(self.first[k]), int(self.count[k]))
                for k in list(range(ns - 1)) + list(range(3 * ns, 4 * ns - 1))]

    def rings_to_m(self, maps):
        """F[f, m, ring] = sum_j x_j e^{-i m phi_j} of (f, npix) maps."""
        nf, ns = maps.shape[0], self.nside
        m = np.arange(self.lmax + 1)
        caps = np.zeros((4 * ns - 1, nf, self.lmax + 1), dtype=np.complex128)
        host = maps.cpu().numpy()
        for k, f, n in self._polar():
            caps[k] = np.fft.fft(host[:, f: f + n])[:, m % n]
        out = torch.from_numpy(caps).to(maps.device).permute(1, 2, 0).contiguous()
        f, n = int(self.first[ns - 1]), 4 * ns
        eq = torch.fft.fft(maps[:, f: f + (2 * ns + 1) * n].reshape(-1, 2 * ns + 1, n))
        out[:, :, ns - 1: 3 * ns] = eq[:, :, m % n].transpose(1, 2)
        return out * self.phase[None]

    def m_to_rings(self, G):
        """Maps (f, npix) of real fields from their G[f, m, ring], m >= 0."""
        H = G * self.phase.conj()[None]
        H[:, 1:] *= 2
        nf, ns = G.shape[0], self.nside
        host = np.zeros((nf, self.npix))
        m = np.arange(self.lmax + 1)
        caps = H.permute(2, 0, 1).contiguous().cpu().numpy()
        for k, f, n in self._polar():
            b = np.zeros((nf, -(-m.size // n) * n), dtype=np.complex128)
            b[:, : m.size] = caps[k]
            host[:, f: f + n] = (np.fft.ifft(b.reshape(nf, -1, n).sum(1)) * n).real
        maps = torch.from_numpy(host).to(G.device)
        f, n = int(self.first[ns - 1]), 4 * ns
        b = torch.zeros(nf, n, 2 * ns + 1, dtype=torch.complex128, device=G.device)
        b[:, : m.size] = H[:, :, ns - 1: 3 * ns]
        eq = (torch.fft.ifft(b, dim=1) * n).real.transpose(1, 2)
        maps[:, f: f + (2 * ns + 1) * n] = eq.reshape(nf, -1)
        return maps

    def _panels(self, spins, width=16):
        """Yields (l0, l1, [harmonics[m, l - l0, ring] for l0 <= l < l1 of each spin])."""
        L, buf = self.lmax, None
        shape = (L + 1, width, self.z.numel())
        for l, vals in self.rows(spins):
            if l % width == 0:
                buf = [torch.zeros(shape, dtype=torch.float64, device=self.z.device) for _ in spins]
            for v, b in zip(vals, buf):
                if v is not None:
                    b[: l + 1, l % width] = v
            if (l + 1) % width == 0 or l == L:
                l0 = l - l % width
                yield l0, l + 1, [b[: l + 1, : l + 1 - l0] for b in buf]

    def _sums(self, F, spins):
        """sum_ring h_lm F[m, c, ring] for the (m, c, ring) columns F[p] of each spin p."""
        L = self.lmax
        out = [torch.zeros(f.shape[1], L + 1, L + 1, dtype=torch.float64, device=f.device)
               for f in F]
        for l0, l1, panels in self._panels(spins):
            for f, h, o in zip(F, panels, out):
                o[:, :l1, l0:l1] = torch.bmm(f[:l1], h.transpose(1, 2)).transpose(0, 1)
        return out

    def _fields(self, cols, spins):
        """G[c, m, ring] = sum_l cols[p][c, m, l] h_lm of each spin p."""
        out = [torch.zeros(self.lmax + 1, c.shape[0], self.z.numel(), dtype=torch.float64,
                           device=c.device) for c in cols]
        for l0, l1, panels in self._panels(spins):
            for c, h, g in zip(cols, panels, out):
                a = c[:, :l1, l0:l1].transpose(0, 1).contiguous()
                g[:l1] += torch.bmm(a, h)
        return [g.transpose(0, 1) for g in out]

    def _columns(self, F):
        """(f, m, ring) complex as (m, 2 f, ring) real."""
        return torch.cat([F.real, F.imag]).transpose(0, 1).contiguous()

    def analyse(self, maps):
        """a[f, m, l] of scalar maps."""
        n = maps.shape[0]
        a = self._sums([self._columns(self.rings_to_m(maps))], (0,))[0]
        return torch.complex(a[:n], a[n:]) * (4 * math.pi / self.npix)

    def synthesise(self, a):
        n = a.shape[0]
        G, = self._fields([torch.cat([a.real, a.imag])], (0,))
        return self.m_to_rings(torch.complex(G[:n].contiguous(), G[n:].contiguous()))

    def analyse_pol(self, Q, U):
        """a_E, a_B [f, m, l] of (f, npix) Q and U maps: _{+-2}Y_lm = N_l d^l_{m,-+2}."""
        n = Q.shape[0]
        FQ, FU = self.rings_to_m(Q), self.rings_to_m(U)
        s = self._sums([self._columns(FQ + 1j * FU), self._columns(FQ - 1j * FU)], (-2, 2))
        a2, am2 = (torch.complex(x[:n], x[n:]) * (4 * math.pi / self.npix) for x in s)
        return -(a2 + am2) / 2, 1j * (a2 - am2) / 2

    def synthesise_pol(self, aE, aB):
        n = aE.shape[0]
        cols = [torch.cat([c.real, c.imag]) for c in (-(aE + 1j * aB), -(aE - 1j * aB))]
        p, m = (torch.complex(g[:n].contiguous(), g[n:].contiguous())
                for g in self._fields(cols, (-2, 2)))
        return self.m_to_rings((p + m) / 2), self.m_to_rings((p - m) / 2j)

    def map2alm(self, maps, niter=3):
        a = self.analyse(maps)
        for _ in range(niter):
            a = a + self.analyse(maps - self.synthesise(a))
        return a

    def map2alm_pol(self, Q, U, niter=3):
        E, B = self.analyse_pol(Q, U)
        for _ in range(niter):
            q, u = self.synthesise_pol(E, B)
            dE, dB = self.analyse_pol(Q - q, U - u)
            E, B = E + dE, B + dB
        return E, B


def _cross(a, b):
    """alm2cl of a[m, l], b[m, l]."""
    x = (a * b.conj()).real
    l = torch.arange(a.shape[1], dtype=torch.float64, device=a.device)
    return (x[0] + 2 * x[1:].sum(0)) / (2 * l + 1)


def _master_exact(case, seed):
    nside, lmin = case["nside"], case["lmin"]
    lmax = 3 * nside - 1
    masks, skies = _masks(nside, 4, seed), _skies(nside, seed)
    sp = _Sphere(nside, lmax)
    m1, m2 = ([s[0] * masks[2 * k], s[1] * masks[2 * k + 1], s[2] * masks[2 * k + 1]]
              for k, s in enumerate(skies))
    a = sp.map2alm(torch.cat([torch.stack([m1[0], m2[0]]), masks]))
    E, B = sp.map2alm_pol(torch.stack([m1[1], m2[1]]), torch.stack([m1[2], m2[2]]))
    w = a[2:]
    W = {x + y: _cross(w["TP".index(x)], w[2 + "TP".index(y)]).cpu().numpy()
         for x in "TP" for y in "TP"}
    alm = {"T": a[:2], "E": E, "B": B}
    p = {x + y: _cross(alm[x][0], alm[y][1])[lmin:] for x in "TEB" for y in "TEB"}
    tt, te, pp, mm = _blocks(lmin, lmax, [("TT", [W["TT"]]), ("TE", [W["TP"], W["PT"]]),
                                          ("M++", [W["PP"]]), ("M--", [W["PP"]])])
    solve = lambda M, *v: torch.linalg.solve(M, torch.stack(v, 1)).T  # noqa: E731
    out = {"TT": solve(tt[0], p["TT"])[0]}
    out["TE"], out["TB"] = solve(te[0], p["TE"], p["TB"])
    out["ET"], out["BT"] = solve(te[1], p["ET"], p["BT"])
    P, M = pp[0], mm[0]
    n = P.shape[0]
    x = solve(torch.cat([torch.cat([P, M], 1), torch.cat([M, P], 1)]), torch.cat([p["EE"], p["BB"]]))[0]
    y = solve(torch.cat([torch.cat([P, -M], 1), torch.cat([-M, P], 1)]),
              torch.cat([p["EB"], p["BE"]]))[0]
    out["EE"], out["BB"], out["EB"], out["BE"] = x[:n], x[n:], y[:n], y[n:]
    return out


def exact(case, seed):
    op = case["op"]
    rng = np.random.default_rng([seed, 0])
    if op == "mcm":
        W = _mask_spectrum(rng, case["lmax"] + 1, case["spec"] == "TE")
        return _blocks(case["lmin"], case["lmax"], [(case["spec"], [W])])[0][0]
    if op == "set":
        tt, te, et, pp = _set_inputs(rng, case["lmax"] + 1)
        b = _blocks(case["lmin"], case["lmax"],
                    [("TT", [tt]), ("TE", [te, et]), ("M++", [pp]), ("M--", [pp])])
        return [x.T.contiguous() for o in b for x in o]
    if op == "cov":
        return _cov_exact(case["kind"], case["lmin"], case["lmax"],
                          *_cov_inputs(rng, case["kind"], case["lmax"] + 1))
    if op == "batch":
        Ws = [_mask_spectrum(rng, case["lmax"] + 1) for _ in range(case["K"])]
        return torch.stack([x.T for x in _blocks(0, case["lmax"], [(case["kind"], Ws)])[0]])
    if op == "mask_spectra":
        a = _Sphere(case["nside"], case["lmax"]).map2alm(_masks(case["nside"], case["nmaps"], seed))
        return torch.stack([torch.stack([_cross(x, y) for y in a]) for x in a])
    if op == "alm2map_pol":
        L, sp = case["lmax"], _Sphere(case["nside"], case["lmax"])
        teb = torch.zeros(3, L + 1, L + 1, dtype=torch.complex128, device=_device())
        m, l = torch.triu_indices(L + 1, L + 1, device=_device())
        teb[:, m, l] = _alms(L, seed)
        I = sp.synthesise(teb[:1])
        Q, U = sp.synthesise_pol(teb[1:2], teb[2:])
        return torch.stack([I[0], Q[0], U[0]])[None]
    if op == "master":
        return _master_exact(case, seed)
    if op == "lu":
        return torch.linalg.solve(*_linear(case, seed))
    if op == "decouple":
        Y, B1, B2 = _linear(case, seed)
        return torch.linalg.solve(B2, torch.linalg.solve(B1, Y).T).T
    res, out = _served_inputs(case, seed), []
    for i, (kind, lmax) in enumerate(_requests(case)):
        n = lmax + 1
        W = [res[(i + k) % 10][:n] for k in range(8)]
        if kind == "PM":
            out.append([x[0] for x in _blocks(0, lmax, [("M++", W[:1]), ("M--", W[:1])])])
        elif kind in KINDS:
            out.append([_blocks(0, lmax, [(kind, W[:1])])[0][0]])
        else:
            nW, nS, nR = COV_ARITY[kind]
            out.append([_cov_exact(kind, 0, lmax, [v[:n] for v in res[10: 10 + nS]],
                                   [v[:n] for v in res[14: 14 + nR]], W[:nW])])
    return out
