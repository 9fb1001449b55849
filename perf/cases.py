"""The work that users of prc_d2z have it do, as cases that can be timed and checked.

Kinds of case (`kind`):
  run      one delta2zreion step on a field that is resident in the context (the
           step that bench.py times): D2Z.run() -> zreion
  field    the step of a loop over realisations: hand over a new device field, run,
           read the per-radius table (R, sigma, sigma_grid) and zreion
  driver   the d2z program's own flow on host arrays: ICs in, zreion out
  group    uneven boxes of one sweep stepped together (Group.run())
  history  the d2z program from its transform to the corrected output: run,
           GetHistory, bubble mean free paths, corrected history, remapped zreion
  power    binned power spectrum of a new device field

Sizes are those of bench.py's workloads and of the tests; cells are about 1.5 to
2 Mpc/h wide, as there.  Fields are Gaussian with a CDM-like spectrum.  Bubble
radii (RecordBubbleSizes) are not among the outputs: the first radius that
reaches a flat maximum is decided by rounding, so two right answers differ by
whole radius steps.  At N = 1024 the radii per batch are set so that several contexts fit one card.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "pr-calc_amd"))

import prc_d2z  # noqa: E402

MODES = {"plain": prc_d2z.PLAIN_FP32, "fused": prc_d2z.FUSED_FP32, "mixed": prc_d2z.FUSED_MIXED,
         "half": prc_d2z.FUSED_HALF}
HOST_COSMOLOGY = dict(Omegam=0.31, Omegab=0.049, Omegal=0.69, h=0.68, ns=0.965, sigma8=0.81, w=-1.0)
ZETA, M_MIN = 40.0, 1.4706e8
GROUP_SIZES = (64, 128, 192, 256)
GROUP_CELL = 1.5625  # Mpc/h


def listed():
    return [
        # the smallest step in use (test-sized box of a parameter sweep): host calls, launches and
        # synchronisations count
        {"name": "field_64_fused", "kind": "field", "mode": "fused", "n": 64, "nscales": 8, "box": 100.0, "rmax": 25.0},
        # the 128^3 x 32 configuration: short kernels back to back
        {"name": "run_128_mixed", "kind": "run", "mode": "mixed", "n": 128, "nscales": 32, "box": 200.0, "rmax": 50.0},
        # the d2z program on host data, a length with a factor 3
        {"name": "driver_192_fused", "kind": "driver", "mode": "fused", "n": 192, "nscales": 24, "box": 300.0,
         "rmax": 50.0},
        # the separate-kernel path in the reference's order
        {"name": "run_256_plain", "kind": "run", "mode": "plain", "n": 256, "nscales": 16, "box": 400.0, "rmax": 50.0},
        # the 512^3 x 64 configuration in the two storage types
        {"name": "run_512_fused", "kind": "run", "mode": "fused", "n": 512, "nscales": 64, "box": 1000.0, "rmax": 80.0},
        {"name": "run_512_half", "kind": "run", "mode": "half", "n": 512, "nscales": 64, "box": 1000.0, "rmax": 80.0},
        # the headline 1024^3 x 96 step, mixed precision and FP16 storage, and a shorter schedule of
        # the FP32 path at the same size
        {"name": "run_1024_mixed", "kind": "run", "mode": "mixed", "n": 1024, "nscales": 96, "box": 2000.0,
         "rmax": 120.0},
        {"name": "run_1024_half", "kind": "run", "mode": "half", "n": 1024, "nscales": 96, "box": 2000.0,
         "rmax": 120.0},
        {"name": "run_1024_fused", "kind": "run", "mode": "fused", "n": 1024, "nscales": 32, "box": 2000.0,
         "rmax": 120.0},
        # uneven boxes together, a quarter of the 48-box workload
        {"name": "group_12_boxes", "kind": "group", "mode": "fused", "n64": 0, "n128": 4, "n192": 4, "n256": 4,
         "nscales": 48, "rmax": 50.0},
        # the whole program after its input: step, history and history correction
        {"name": "history_256_plain", "kind": "history", "mode": "plain", "n": 256, "nscales": 8, "box": 400.0,
         "rmax": 50.0},
        # analysis of a field: forward transform and binning
        {"name": "power_512", "kind": "power", "mode": "fused", "n": 512, "nscales": 2, "box": 1000.0, "rmax": 80.0,
         "nk": 60},
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "field", "driver", "group", "history", "power"])
    cell = rng.uniform(1.4, 2.1)
    if kind == "group":
        c = {"kind": kind, "mode": "fused", "n64": rng.randint(0, 5), "n128": rng.randint(0, 5),
             "n192": rng.randint(0, 3), "n256": rng.randint(1, 3), "nscales": _loguniform(rng, 5, 48)}
        c["rmax"] = round(rng.uniform(20.0, 25.0), 2)
        return c
    if kind == "run":
        mode = rng.choice(["plain", "fused", "mixed", "half"])
        n = rng.choice([32, 64, 128, 192, 256, 512, 1024] if mode != "plain" else [32, 64, 128, 192, 256, 512])
        ns = _loguniform(rng, 4, 96 if mode != "plain" else 40)
    elif kind == "field":
        mode, n, ns = rng.choice(["fused", "mixed", "half"]), rng.choice([32, 64, 128, 192, 256]), _loguniform(rng, 4, 40)
    elif kind == "driver":
        mode, n, ns = rng.choice(["fused", "plain"]), rng.choice([64, 128, 192, 256]), _loguniform(rng, 4, 40)
    elif kind == "history":
        mode, n, ns = "plain", rng.choice([128, 192, 256]), _loguniform(rng, 4, 16)
    else:
        mode, n, ns = "fused", rng.choice([64, 128, 192, 256, 512]), 2
    box = round(cell * n, 2)
    c = {"kind": kind, "mode": mode, "n": n, "nscales": ns, "box": box,
         "rmax": round(min(120.0, box * rng.uniform(0.12, 0.25)), 2)}
    if kind == "power":
        c["nk"] = rng.randint(15, 200)
    return c


# ------------------------------------------------------------------ inputs
def _field(n, box, seed):
    """Gaussian density contrast [n][n][n], FP32 on the GPU, made from the seed alone: white noise
    coloured by sqrt(P), P = k^ns T(k)^2 with the BBKS transfer function of Gamma = 0.2."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    f = torch.randn((n, n, n), generator=g, device="cuda", dtype=torch.float32)
    s = torch.fft.rfftn(f)
    del f
    dk = 2.0 * math.pi / box
    fx = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    fz = torch.fft.rfftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    for x in range(n):
        k = torch.sqrt(fx[x] ** 2 + fx[:, None] ** 2 + fz[None, :] ** 2) * dk
        q = (k / 0.2).clamp_min(1e-9)
        t = torch.log1p(2.34 * q) / (2.34 * q) * (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 +
                                                  (6.71 * q) ** 4) ** -0.25
        amp = torch.where(k > 0, k ** 0.4825 * t, torch.zeros_like(k))
        s[x] *= amp.float()
    f = torch.fft.irfftn(s, s=(n, n, n))
    del s
    # rms of the linear field at z = 0 in cells of this width
    f *= 2.4 * (1.5625 * n / box) ** 0.55 / f.square().mean(dtype=torch.float64).sqrt().float()
    return f


class _DeviceArray:
    """A device buffer of a context, for torch; the tensor holds this object, and it the context, whose
    end frees the buffer."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _zreion_of(d):
    return torch.as_tensor(_DeviceArray(d, d.zreion_device_ptr(), (d.N, d.N, d.N)), device="cuda")


def _params(c, n, box):
    # at 1024^3 a batch of 16 FP32 radii (32 in FP16 storage) takes 69 GB of intermediates
    rpl = 16 if n == 1024 and c["mode"] != "half" else 0
    return prc_d2z.D2ZParams(N=n, Nscales=c["nscales"], BoxSize=box, Rmax=c["rmax"], zeta=ZETA, M_min=M_MIN,
                             mode=MODES[c["mode"]], radii_per_launch=rpl, **HOST_COSMOLOGY)


def _context(c, n, box):
    d = prc_d2z.D2Z(_params(c, n, box))
    if c["mode"] == "mixed" and n == 1024:
        # the plans that the autotuner picks there, set directly as a program that keeps them does
        d.set_plan(prc_d2z.PLAN_MATRIX, prc_d2z.PLAN_VECTOR, 16)
    return d


def _boxes(c):
    return [(n, n * GROUP_CELL) for n in GROUP_SIZES for _ in range(c["n%d" % n])]


def _fcoll_table():
    z = np.arange(2000) * (50.0 / 2000)
    return (0.03 * np.exp(-((z / 9.0) ** 2))).astype(np.float32)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "group":
        boxes = []
        for k, (n, box) in enumerate(_boxes(c)):
            f = _field(n, box, seed + 1000 * k)
            torch.cuda.synchronize()  # the contexts have streams of their own
            d = _context(c, n, box)
            d.set_delta_device(f.data_ptr())
            boxes.append(d)
        group = prc_d2z.Group(boxes)
        return {"kind": kind, "group": group, "zreion": [_zreion_of(d) for d in boxes], "boxes": boxes}
    n, box = c["n"], c["box"]
    f = _field(n, box, seed)
    torch.cuda.synchronize()
    if kind == "driver":
        host = f.cpu().numpy()
        del f
        return {"kind": kind, "d": _context(c, n, box), "delta": host}
    if n == 1024:
        torch.cuda.empty_cache()  # the transforms' scratch
    d = _context(c, n, box)
    state = {"kind": kind, "d": d, "zreion": _zreion_of(d)}
    if kind in ("field", "power"):
        state["delta"] = f
        if kind == "power":
            dk = 2.0 * math.pi / box
            state["bins"] = (c["nk"], 0.5 * dk, 0.9 * dk * n)
    else:
        d.set_delta_device(f.data_ptr())
        del f
        if n == 1024:
            torch.cuda.empty_cache()
        if kind == "history":
            state["fcoll"] = _fcoll_table()
    return state


# -------------------------------------------------------------------- pass
def run(state):
    kind = state["kind"]
    if kind == "group":
        state["group"].run()
        return state["zreion"]
    d = state["d"]
    if kind == "run":
        d.run()
        return {"zreion": state["zreion"]}
    if kind == "field":
        d.set_delta_device(state["delta"].data_ptr())
        d.run()
        return {"table": d.radius_table(), "zreion": state["zreion"]}
    if kind == "driver":
        d.set_delta(state["delta"])
        d.run()
        return {"zreion": d.zreion()}
    if kind == "power":
        d.set_delta_device(state["delta"].data_ptr())
        nk, kmin, kmax = state["bins"]
        p = d.power_spectrum(nk, kmin, kmax)
        return {"ps": p["ps"], "ook2": p["ook2"], "kmean": p["kmean"], "nmodes": p["nmodes"]}
    d.run()
    counts = d.history()
    hist = d.cumulative_history(counts, d.N)
    mfp, mfp_x, dfdmfp = d.bubble_mfp(hist, seed=1)
    ch = d.corrected_history(state["fcoll"], 0.0, 50.0, mfp)
    d.correct_zreion(hist, ch)
    return {"chistory": ch, "corrected": state["zreion"], "counts": counts.astype(np.int64), "dfdmfp": dfdmfp,
            "mfp": mfp}


def work(case):
    """Bytes: every input read once, every output written once.  Flops: 2.5 M log2 M for a real
    transform of M cells, the filter on the half spectrum and the barrier on every cell."""
    def step(n, nscales):
        m = float(n) ** 3
        fft = 2.5 * m * math.log2(m)
        return {"bytes": 8.0 * m, "flops": fft + nscales * (fft + 6.0 * m)}

    kind = case["kind"]
    if kind == "group":
        each = [step(n, case["nscales"]) for n, _ in _boxes(case)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    w = step(case["n"], case["nscales"])
    m = float(case["n"]) ** 3
    if kind == "history":  # the histogram's read and the remap's read and write, 4e7 skewers' cells
        w["bytes"] += 12.0 * m + 4.0 * 4e7
    elif kind == "power":
        w = {"bytes": 4.0 * m, "flops": 2.5 * m * math.log2(m) + 10.0 * m / 2}
    return w


# ------------------------------------------------------- the same in 64 bits
# FP32 where the d2z program's own definitions are FP32 (its parameters and its radii,
# delta2zreion_d2z.C:36-38,55), FP64 elsewhere.
def _radii(c, n, box):
    f = np.float32
    h = f(HOST_COSMOLOGY["h"])
    l0 = f(math.log10(float(f(f(f(box) / h) * f(1.0)) / f(n))))
    l1 = f(math.log10(float(f(f(c["rmax"]) / h))))
    dl = f(f(l1 - l0) / f(c["nscales"] - 1))
    return np.array([f(10.0 ** float(f(l0 + f(f(r) * dl)))) for r in range(c["nscales"])], dtype=np.float64)


def _sigma2(R):
    """Unnormalised sigma^2 of the Eisenstein & Hu (1998) no-wiggle spectrum, top-hat radius R [Mpc]."""
    om, ob, hh, an = (float(np.float32(HOST_COSMOLOGY[k])) for k in ("Omegam", "Omegab", "h", "ns"))
    x, w = np.polynomial.legendre.leggauss(8)
    a, b, panels = math.log(1e-5 / R), math.log(1e5 / R), 4096
    hw = 0.5 * (b - a) / panels
    k = np.exp(a + hw * (2 * np.arange(panels)[:, None] + 1) + hw * x[None, :])
    alpha = 1 - 0.328 * math.log(431 * om * hh * hh) * (ob / om) + 0.38 * math.log(22.3 * om * hh * hh) * (ob / om) ** 2
    sound = 44.5 * math.log(9.83 / (om * hh * hh)) / math.sqrt(1 + 10 * (ob * hh * hh) ** 0.75)
    q = (k / hh) * (2.728 / 2.7) ** 2 / (om * hh * (alpha + (1 - alpha) / (1 + (0.43 * k * sound) ** 4)))
    lg = np.log(2 * math.e + 1.8 * q)
    t = lg / (lg + (14.2 + 731 / (1 + 62.5 * q)) * q * q)
    kr = k * R
    win = 3 * (np.sin(kr) - kr * np.cos(kr)) / kr ** 3
    return float(np.sum(w * k ** (3 + an) * t * t * win * win) * hw)


def _growth(z):
    """Linear growth factor, the Carroll, Press & Turner (1992) fit for w = -1."""
    om, ol = float(np.float32(HOST_COSMOLOGY["Omegam"])), float(np.float32(HOST_COSMOLOGY["Omegal"]))

    def g(o, lam):
        return 2.5 * o / (o ** (4.0 / 7.0) - lam + (1 + o / 2) * (1 + lam / 70))

    x = 1.0 + z
    e = om * x ** 3 + (1 - om - ol) * x ** 2 + ol
    return g(om * x ** 3 / e, ol / e) / x / g(om, ol)


def _inverse_erfc(y):
    """The d2z program's root of erfc(t) = y: Brent's method (Brent 1973, ch. 4) on [0, 100] until the
    bracket is within 1e-4 of its lower end, which is the answer (math.C:23-61)."""
    def f(t):
        return math.erfc(t) - y

    eps = np.finfo(float).eps
    a, b = 0.0, 100.0
    fa, fb = f(a), f(b)
    c, fc, d, e = b, fb, b - a, b - a
    for _ in range(100):
        secant = False
        if fb * fc > 0:
            secant, c, fc, d, e = True, a, fa, b - a, b - a
        if abs(fc) < abs(fb):
            secant, a, b, c, fa, fb, fc = True, b, c, b, fb, fc, fb
        tol, m = 0.5 * eps * abs(b), 0.5 * (c - b)
        if fb == 0:
            return b
        if abs(m) <= tol:
            return min(b, c)
        if abs(e) < tol or abs(fa) <= abs(fb):
            d = e = m
        else:
            s = fb / fa
            if secant:
                p, q = 2 * m * s, 1 - s
            else:
                q, r = fa / fc, fb / fc
                p, q = s * (2 * m * q * (q - r) - (b - a) * (r - 1)), (q - 1) * (r - 1) * (s - 1)
            p, q = abs(p), (-q if p > 0 else q)
            if 2 * p < min(3 * m * q - abs(tol * q), abs(e * q)):
                d, e = p / q, d
            else:
                d = e = m
        a, fa = b, fb
        b += d if abs(d) > tol else math.copysign(tol, m)
        fb = f(b)
        if fb * fc > 0:
            c = a
        lo, hi = min(b, c), max(b, c)
        if lo > 0 and hi - lo < 1e-4 * lo:
            return lo
    return lo


def _exact_step(c, n, box, seed):
    """zreion and the per-radius table, from the field in FP64."""
    om, h, s8 = (float(np.float32(HOST_COSMOLOGY[k])) for k in ("Omegam", "h", "sigma8"))
    pn2 = s8 * s8 / _sigma2(8.0 / h)
    dens = 2.775e11 * om * h * h
    smin2 = pn2 * _sigma2((3 * float(np.float32(M_MIN)) / (4 * float(np.float32(math.pi))) / dens) ** (1 / 3))
    R = _radii(c, n, box)
    # the program's mass of a radius and back, its pi in FP32
    pi = float(np.float32(math.pi))
    sig2 = np.array([pn2 * _sigma2((math.pi / pi) ** (1 / 3) * r) for r in R])
    erfz = _inverse_erfc(float(np.float32(1.0 / ZETA)))
    A = 21.0 * _growth(20.0) / float(np.float32(1.686))
    s = torch.fft.rfftn(_field(n, box, seed).double() / _growth(0.0))
    fx = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    fz = torch.fft.rfftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
    # dk of the d2z program (float), |k| per plane of the spectrum
    dk = float(np.float32(2.0 * math.pi / float(np.float32(box) / np.float32(h))))
    zre = torch.zeros((n, n, n), device="cuda", dtype=torch.float64)
    grid = []
    # W by |k|^2 in units of dk^2, an integer
    m2 = (fx[:, None, None] ** 2 + fx[None, :, None] ** 2 + fz[None, None, :] ** 2).int()
    k = torch.arange(3 * (n // 2) ** 2 + 1, device="cuda", dtype=torch.float64).sqrt() * dk
    m = torch.empty_like(s)
    for r, s2 in zip(R, sig2):
        kr = k * r
        w = torch.where(kr < 1e-2, 1 - kr ** 2 / 10 + kr ** 4 / 280,
                        3 * (torch.sin(kr) - kr * torch.cos(kr)) / kr ** 3)
        w[0] = 0.0
        torch.mul(s, w[m2], out=m)
        d = torch.fft.irfftn(m, s=(n, n, n))
        if c["kind"] == "field":
            grid.append(float(d.square().mean().sqrt()))
        if s2 > smin2:
            continue
        z = d.add_(math.sqrt(2 * (smin2 - s2)) * erfz).mul_(A).sub_(1.0)
        torch.maximum(zre, z, out=zre)
        del d, z
    out = {"zreion": zre}
    if grid:
        out["table"] = np.stack([R * h, np.sqrt(sig2), np.array(grid)], axis=1)
    return out


def _exact_power(c, seed):
    """Binned power of the field in FP64; the bin of a mode by the reference's FP32 wave number."""
    n, nk, box = c["n"], c["nk"], c["box"]
    s = torch.fft.rfftn(_field(n, box, seed).double())
    dk0 = 2.0 * math.pi / box
    kmin, kmax = np.float32(0.5 * dk0), np.float32(0.9 * dk0 * n)
    dk = np.float32(2.0 * math.pi / float(np.float32(box)))
    lmin = np.float32(math.log(float(kmin)))
    dl = np.float32((np.float32(math.log(float(kmax))) - lmin) / np.float32(nk))
    i = torch.arange(n, device="cuda", dtype=torch.float32) * float(dk)
    kg = float(np.float32(dk * np.float32(n)))
    f = torch.where(torch.arange(n, device="cuda") >= n // 2, i - kg, i)
    fz = f[:n // 2 + 1]
    sums = [torch.zeros(nk, device="cuda", dtype=torch.float64) for _ in range(4)]
    scale = 1.0 / float(n) ** 3 / float(np.float32(kg)) ** 3
    for x in range(n):
        k2 = f[x] ** 2 + f[:, None] ** 2 + fz[None, :] ** 2
        k = torch.sqrt(k2)
        u = (torch.log(k) - float(lmin)) / float(dl)
        ok = (u > -1.0) & (u < nk)
        b = u[ok].int().long()
        p = s[x][ok]
        vals = (torch.ones_like(b, dtype=torch.float64), (p.real ** 2 + p.imag ** 2) * scale, 1.0 / k2[ok].double(),
                k[ok].double())
        for t, v in zip(sums, vals):
            t.index_add_(0, b, v)
    cnt, ps, ook2, km = (t.cpu().numpy() for t in sums)
    with np.errstate(invalid="ignore", divide="ignore"):
        return {"ps": ps * (2 * math.pi) ** 3 / cnt, "ook2": ook2 / cnt, "kmean": km / cnt, "nmodes": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "history":
        return None  # Monte Carlo walks on thresholds of the field
    if kind == "power":
        return _exact_power(case, seed)
    if kind == "group":
        return [_exact_step(case, n, box, seed + 1000 * k)["zreion"] for k, (n, box) in enumerate(_boxes(case))]
    return _exact_step(case, case["n"], case["box"], seed)
