"""The work that users of the likelihood have it do, as measurable cases.

A case is one observed system (or several) and one call of a public entry
point on it: `loglike` (one candidate, the callback a sampler calls),
`batch` (many candidates of one system, the batched sampler's call),
`systems` (physical parameters of several systems of uneven size in one
launch) or `render` (the planes of one parameter vector, written when the
sampler reports progress).  Flags are those the command line sets: batched
calls replay a captured graph, `table` is the tabulated EPL lens.

Fields of a case: entry, lens (object name), sources (object names joined by
"+"; "sky" is a foreground), width, height, einstein (the lens scale in
pixels), psf ("none", "gauss", "moffat") with psfw x psfh taps, rule,
candidates, table, spread (1: unit-cube draws, as early in a run; less: draws
from a box of that width around the truth, as later in a run), mix (for
`systems`: how many systems; their sizes follow from the case alone).
"""
import math
import random

import numpy as np
import torch

from lensed_amd import workloads as W
from lensed_amd._lib import LENSED_GRAPH, LENSED_TABLE
from lensed_amd.lensed import Context, SystemSpec

SIGMA = 0.05  # noise per pixel; the data's brightest pixel is ten of these

BASE = {"entry": "batch", "lens": "sie", "sources": "sersic", "width": 100, "height": 100, "einstein": 20.0,
        "psf": "none", "psfw": 0, "psfh": 0, "rule": "g3k7", "candidates": 256, "table": False, "spread": 1.0,
        "mix": 0}


def _case(name, **fields):
    return {"name": name, **BASE, **fields}


def listed():
    epl = {"lens": "epl_plus_shear", "sources": "gauss", "width": 256, "height": 256, "psf": "gauss", "psfw": 21,
           "psfh": 21, "table": True}
    disk = {"lens": "epl_plus_shear", "sources": "sersic+sersic+sky", "width": 512, "height": 512, "einstein": 40.0,
            "psf": "moffat", "psfw": 31, "psfh": 31}
    return [
        # the sampler's plain callback on the smallest system: latency
        _case("loglike-100", entry="loglike", candidates=1),
        # the same callback on a full cutout with a PSF and the tabulated lens
        _case("loglike-256-table", entry="loglike", candidates=1, **epl),
        # the progress report: model, quadrature error, convolved image and chi^2 planes of one point
        _case("render-512", entry="render", candidates=1, **disk),
        # the smallest launch of the batched sampler
        _case("batch-100x256"),
        # bulge, disk and sky behind a sheared lens, a full launch
        _case("batch-200x1024", lens="sie_plus_shear", sources="sersic+exponential+sky", width=200, height=200,
              psf="gauss", psfw=21, psfh=21, candidates=1024),
        # the tabulated lens: the sampler's smallest launch late in a run, and the full launch over the prior
        _case("batch-256x256-late", candidates=256, spread=0.2, **epl),
        _case("batch-256x4096", candidates=4096, **epl),
        # the same system with the lens's series per ray, the command line's default
        _case("batch-256x512-series", candidates=512, **{**epl, "table": False}),
        # a follow-up fit: two Sersic components on a large cutout, a PSF of high rank
        _case("batch-512x512", candidates=512, spread=0.5, **{**disk, "table": True}),
        # a cored lens on an odd cutout, a narrow and tall PSF, a count no power of two
        _case("batch-131x97-odd", lens="nsie", sources="exponential", width=131, height=97, einstein=11.0,
              psf="gauss", psfw=15, psfh=9, candidates=333),
        # a survey's systems of 64 to 512 pixels in one launch
        _case("systems-16x64", entry="systems", mix=16, candidates=64, einstein=0.0),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    c = dict(BASE)
    c["entry"] = rng.choice(["batch"] * 7 + ["loglike", "render", "systems"])
    c["lens"] = rng.choice(["sie", "sie_plus_shear", "nsie", "epl", "epl_plus_shear", "epl_plus_shear"])
    c["sources"] = rng.choice(["gauss", "gauss", "sersic", "exponential", "sersic+sky", "sersic+sersic+sky",
                               "sersic+exponential+sky"])
    c["width"] = log_int(48, 512)
    c["height"] = min(512, max(48, int(c["width"] * rng.uniform(0.7, 1.4))))
    n = min(c["width"], c["height"])
    c["einstein"] = round(n * rng.uniform(0.07, 0.18), 2)
    c["psf"] = rng.choice(["none", "gauss", "gauss", "gauss", "moffat"])
    if c["psf"] != "none":
        c["psfw"] = 2 * rng.randint(3, 15) + 1
        c["psfh"] = c["psfw"] if rng.random() < 0.7 else 2 * rng.randint(3, 15) + 1
    c["rule"] = rng.choice(["g3k7", "g3k7", "g3k7", "sub4"])
    c["table"] = c["lens"].startswith("epl") and rng.random() < 0.7
    c["spread"] = rng.choice([1.0, 1.0, 0.3])
    most = 4096
    if c["entry"] in ("loglike", "render"):
        most = 1
    elif c["entry"] == "systems":
        c["mix"] = rng.randint(2, 12)
        c["width"] = c["height"] = c["psfw"] = c["psfh"] = 0
        c["lens"], c["sources"], c["psf"], c["table"], c["rule"] = "sie", "sersic", "none", False, "g3k7"
        c["einstein"] = round(rng.uniform(0, 1), 3)  # no two mixes alike
        most = 64
    else:
        # no more rays than the largest listed case that traces all of them
        most = min(most, max(1, 80_000_000 // (c["width"] * c["height"])))
    c["candidates"] = min(most, log_int(1, most) if c["entry"] == "systems" else log_int(min(64, most), most))
    return c


# ------------------------------------------------------------------- inputs

PARAMS = {
    "sie": ("x", "y", "r", "q", "pa"),
    "sie_plus_shear": ("x", "y", "r", "q", "pa", "g1", "g2"),
    "nsie": ("x", "y", "r", "rc", "q", "pa"),
    "epl": ("x", "y", "r", "t", "q", "pa"),
    "epl_plus_shear": ("x", "y", "r", "t", "q", "pa", "g1", "g2"),
    "gauss": ("x", "y", "sigma", "mag", "q", "pa"),
    "sersic": ("x", "y", "r", "mag", "n", "q", "pa"),
    "exponential": ("x", "y", "rs", "mag", "q", "pa"),
    "sky": ("bg", "dx", "dy"),
}


def _systems(case):
    """The (lens, sources, width, height, einstein, psf, psfw, psfh) of each system."""
    if case["entry"] != "systems":
        return [(case["lens"], case["sources"].split("+"), case["width"], case["height"], case["einstein"],
                 case["psf"], case["psfw"], case["psfh"])]
    rng = random.Random("%s %s" % (case["mix"], case["einstein"]))
    out = []
    for _ in range(case["mix"]):
        n, k = rng.choice([64, 128, 256, 512]), rng.choice([15, 31])
        out.append((rng.choice(["sie", "epl"]), ["sersic"], n, n, n / 8, "gauss", k, k))
    return out


def _psf(kind, w, h):
    if kind == "none":
        return None
    n = max(w, h)
    p = W.gaussian_psf(n, 3.0) if kind == "gauss" else W.moffat_psf(n, 3.0, 3.0)
    p = p[(n - h) // 2:(n - h) // 2 + h, (n - w) // 2:(n - w) // 2 + w]
    return np.ascontiguousarray(p / p.sum(), dtype=np.float32)


def _ranges(system):
    """(objects, {id.parameter: (lower, upper)}) of one system's priors."""
    lens, sources, w, h, r, _, _, _ = system
    cx, cy = (w + 1) / 2, (h + 1) / 2
    span = {
        "lens": {"x": (cx - 2, cx + 2), "y": (cy - 2, cy + 2), "r": (0.8 * r, 1.2 * r), "rc": (0.02 * r, 0.2 * r),
                 "t": (0.5, 1.5), "q": (0.4, 0.95), "pa": (0, 180), "g1": (-0.1, 0.1), "g2": (-0.1, 0.1)},
        "source": {"x": (cx - 4, cx + 4), "y": (cy - 4, cy + 4), "r": (0.1 * r, 0.4 * r), "rs": (0.1 * r, 0.3 * r),
                   "sigma": (0.075 * r, 0.125 * r), "mag": (-5, 5), "n": (1, 4), "q": (0.4, 1), "pa": (0, 180)},
        "sky": {"bg": (-0.1, 0.1), "dx": (0, 0), "dy": (0, 0)},
    }
    objects, ranges = [("lens", lens)], {}
    for i, s in enumerate(sources):
        objects.append(("sky" if s == "sky" else "source%d" % i, s))
    for oid, name in objects:
        for p in PARAMS[name]:
            ranges["%s.%s" % (oid, p)] = span["lens" if oid == "lens" else "sky" if name == "sky" else "source"][p]
    return objects, ranges


def _inputs(case, seed):
    """Per system: objects, ranges, data, PSF, the free parameters, candidates
    as unit cubes and as physical parameters (object order)."""
    out = []
    for k, system in enumerate(_systems(case)):
        rng = np.random.default_rng([seed, k])
        _, _, w, h, _, kind, pw, ph = system
        objects, ranges = _ranges(system)
        lo = np.array([v[0] for v in ranges.values()], float)
        hi = np.array([v[1] for v in ranges.values()], float)
        free = hi > lo
        u = rng.uniform(0.3, 0.7, len(lo))
        truth = lo + u * (hi - lo)
        psf = _psf(kind, pw, ph)
        # mock data: the model of the truth at one ray per pixel, its sources
        # scaled so that the brightest pixel is ten noise sigmas
        mags = [i for i, p in enumerate(ranges) if p.endswith(".mag")]
        truth[mags] = 0.0
        dim = truth.copy()
        for i, p in enumerate(ranges):
            if p.endswith(".bg"):
                dim[i] = 0.0
        peak = float(_model(objects, torch.tensor(dim[None]), w, h, psf, "point")[0].max())
        shift = -2.5 * math.log10(10 * SIGMA / peak)
        truth[mags] = shift
        lo[mags], hi[mags] = lo[mags] + shift, hi[mags] + shift
        u[mags] = 0.5
        model = _model(objects, torch.tensor(truth[None]), w, h, psf, "point")[0].cpu().numpy()
        image = (model + rng.normal(0, SIGMA, (h, w))).astype(np.float32)
        weight = np.full((h, w), 1 / SIGMA ** 2, np.float32)
        weight[rng.random((h, w)) < 0.01] = 0  # masked pixels
        n = case["candidates"]
        s = case["spread"]
        base = np.clip(u[free] - s / 2, 0, 1 - s)
        cubes = base + s * rng.random((n, int(free.sum())))
        phys = np.tile(lo, (n, 1))
        phys[:, free] = lo[free] + cubes * (hi - lo)[free]
        out.append({"objects": objects, "names": list(ranges), "lo": lo, "hi": hi, "free": free, "image": image,
                    "weight": weight, "psf": psf, "cubes": cubes, "phys": phys})
    return out


def _flags(case):
    many = case["entry"] in ("batch", "systems")
    return (LENSED_GRAPH if many else 0) | (LENSED_TABLE if case["table"] else 0)


def prepare(case, seed):
    specs, inputs = [], _inputs(case, seed)
    for s in inputs:
        priors = {}
        for name, lo, hi, free in zip(s["names"], s["lo"], s["hi"], s["free"]):
            priors[name] = "unif %r %r" % (float(lo), float(hi)) if free else repr(float(lo))
        specs.append(SystemSpec(s["objects"], priors, s["image"], s["weight"], psf=s["psf"], rule=case["rule"]))
    context = Context(specs, flags=_flags(case), max_batch=case["candidates"])
    return {"entry": case["entry"], "context": context, "cubes": inputs[0]["cubes"],
            "phys": [s["phys"] for s in inputs]}


def run(state):
    context, entry = state["context"], state["entry"]
    if entry == "loglike":
        logl, params = context.loglike(state["cubes"][0])
        return {"logl": logl, "params": params}
    if entry == "batch":
        logl, params = context.loglike_batch(state["cubes"])
        return {"logl": logl, "params": params}
    if entry == "systems":
        return {"logl": context.loglike_phys(state["phys"])}
    return context.render(state["phys"][0][0])


# --------------------------------------------------------------------- work

# operations per ray: add, multiply, divide 1, fused multiply-add 2,
# transcendental 1, as the objects' formulas have them
RAY = {"sie": 25, "sie_plus_shear": 31, "nsie": 27, "epl": 120, "epl_plus_shear": 128, "gauss": 14, "sersic": 18,
       "exponential": 16, "sky": 5}
NODES = {"point": 1, "sub4": 16, "g3k7": 49}


def work(case):
    n, flops, nbytes = case["candidates"], 0.0, 0.0
    for lens, sources, w, h, _, kind, pw, ph in _systems(case):
        ray = RAY[lens] + sum(RAY[s] for s in sources)
        if case["table"]:
            ray -= 90  # the angular series once per candidate instead of per ray
        share = 1.0
        if case["table"] and sources == ["gauss"]:
            share = 0.16  # a Gaussian is below single precision's range over most of the image
        taps = 0 if kind == "none" else 2 * (pw + ph) if kind == "gauss" else 2 * pw * ph
        flops += n * w * h * (share * (NODES[case["rule"]] * ray + taps) + 4)
        npar = sum(len(PARAMS[o]) for o in [lens] + sources)
        nbytes += w * h * 8 + pw * ph * 4 + n * (2 * npar + 1) * 8
        if case["entry"] == "render":
            nbytes += 4 * 4 * w * h
    return {"bytes": nbytes, "flops": flops}


# -------------------------------------------------------------------- exact

# Kronrod's 7-point extension of the 3-point Gauss rule on [-1, 1]
K7 = ((0.960491268708020283423507092629080, 0.104656226026467265193823857192073),
      (0.774596669241483377035853079956480, 0.268488089868333440728569280666710),
      (0.434243749346802558002071502844628, 0.401397414775962222905051818618432))
K7_MID = 0.450916538658474142345110087045571


def _nodes(rule):
    """(offset, weight) along one axis of the unit pixel; the rules are products."""
    if rule == "point":
        return [(0.0, 1.0)]
    if rule == "sub4":
        return [(-0.375 + 0.25 * i, 0.25) for i in range(4)]
    return [(0.5 * s * x, 0.5 * w) for x, w in K7 for s in (-1, 1)] + [(0.0, 0.5 * K7_MID)]


def _rotate(par, x, y):
    a = par["pa"] * (math.pi / 180)
    c, s = torch.cos(a), torch.sin(a)
    dx, dy = x - par["x"], y - par["y"]
    return c, s, c * dx + s * dy, c * dy - s * dx


def _deflect(name, par, x, y):
    c, s, u, v = _rotate(par, x, y)
    q = par["q"]
    if name.startswith("epl"):
        # n |z|^(1-t) times the angular series to tenth order (Tessore & Metcalf 2015)
        scale = par["r"] * torch.sqrt(q)
        u, v = q * u / scale, v / scale
        rr = torch.sqrt(u * u + v * v)
        e = torch.complex(u / rr, v / rr)
        z = e * e
        f, T = (1 - q) / (1 + q), 2 - par["t"]
        coef = [torch.ones_like(q)]
        for k in range(1, 11):
            coef.append(coef[-1] * (-f * (2 * k - T) / (2 * k + T)))
        p = coef[10].to(torch.complex128)
        for k in range(9, -1, -1):
            p = p * z + coef[k]
        p = p * e * (2 * scale / (1 + q) * rr ** (1 - par["t"]))
        ax, ay = p.real, p.imag
    else:
        ecc = torch.sqrt(1 - q * q)
        w = torch.sqrt(q * q * u * u + v * v)
        core = par["rc"] if name == "nsie" else 0.0
        amp = par["r"] * torch.sqrt(q) / ecc
        ax, ay = amp * torch.atan(ecc * u / (core + w)), amp * torch.atanh(ecc * v / (core * q * q + w))
    ax, ay = c * ax - s * ay, s * ax + c * ay
    if name.endswith("_plus_shear"):
        dx, dy = x - par["x"], y - par["y"]
        ax, ay = ax + par["g1"] * dx + par["g2"] * dy, ay + par["g2"] * dx - par["g1"] * dy
    return ax, ay


def _brightness(name, par, x, y):
    _, _, u, v = _rotate(par, x, y)
    q, lum = par["q"], 10 ** (-0.4 * par["mag"])
    uu = q * q * u * u + v * v
    if name == "gauss":
        sg = par["sigma"]
        return lum / (2 * math.pi * sg * sg * q) * torch.exp(-0.5 * uu / (sg * sg))
    if name == "exponential":
        rs = par["rs"]
        return lum / (2 * math.pi * rs * rs * q) * torch.exp(-torch.sqrt(uu) / rs)
    n, r = par["n"], par["r"]  # Sersic, b(n) from Ciotti & Bertin's series
    b = 2 * n - 1 / 3 + 4 / (405 * n) + 46 / (25515 * n ** 2) + 131 / (1148175 * n ** 3) \
        - 2194697 / (30690717750 * n ** 4)
    lnorm = -0.4 * math.log(10) * par["mag"] + 2 * n * torch.log(b) - math.log(math.pi) - 2 * torch.log(r) \
        - torch.lgamma(2 * n + 1)
    return torch.exp(lnorm - b * (uu / (q * r * r)) ** (0.5 / n))


def _model(objects, phys, w, h, psf, rule):
    """Convolved model images [K, h, w] of parameters [K, npar], in 64 bits."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    phys = phys.to(dev, torch.float64)
    pars, at = [], 0
    for _, name in objects:
        pars.append((name, {p: phys[:, at + i, None, None] for i, p in enumerate(PARAMS[name])}))
        at += len(PARAMS[name])
    gx = torch.arange(1, w + 1, device=dev, dtype=torch.float64)[None, None, :]
    gy = torch.arange(1, h + 1, device=dev, dtype=torch.float64)[None, :, None]
    f = torch.zeros((phys.shape[0], h, w), device=dev, dtype=torch.float64)
    for ox, wx in _nodes(rule):
        for oy, wy in _nodes(rule):
            x, y = gx + ox, gy + oy
            ax, ay = _deflect(*pars[0], x, y)
            ok = torch.isfinite(ax) & torch.isfinite(ay)
            sx, sy = torch.where(ok, x - ax, -1e10), torch.where(ok, y - ay, -1e10)
            for name, par in pars[1:]:
                if name == "sky":
                    f += wx * wy * (par["bg"] + par["dx"] * (x - 1) + par["dy"] * (y - 1))
                else:
                    f += wx * wy * _brightness(name, par, sx, sy)
    return f if psf is None else _convolve(f, psf)


def _convolve(f, psf):
    """The flipped PSF over the image, its border rows and columns repeated."""
    (ph, pw), (_, h, w) = psf.shape, f.shape
    dev = f.device
    rows = torch.arange(h + ph - 1, device=dev).sub(ph // 2).clamp(0, h - 1)
    cols = torch.arange(w + pw - 1, device=dev).sub(pw // 2).clamp(0, w - 1)
    g = f[:, rows][:, :, cols]
    out = torch.zeros_like(f)
    for j in range(ph):
        for i in range(pw):
            out.add_(g[:, ph - 1 - j:ph - 1 - j + h, pw - 1 - i:pw - 1 - i + w], alpha=float(psf[j, i]))
    return out


def exact(case, seed):
    rays = sum(s[2] * s[3] for s in _systems(case)) * case["candidates"] * NODES[case["rule"]]
    if rays > 1.5e10:
        return None
    inputs = _inputs(case, seed)
    if case["entry"] == "render":
        s = inputs[0]
        h, w = s["image"].shape
        phys = torch.tensor(s["phys"][:1])
        value = _model(s["objects"], phys, w, h, None, case["rule"])
        image = value if s["psf"] is None else _convolve(value, s["psf"])
        data, weight = torch.tensor(s["image"], device=image.device), torch.tensor(s["weight"], device=image.device)
        chi2 = weight.double() * (image[0] - data.double()) ** 2
        return {"value": value[0].cpu().numpy(), "error": None, "image": image[0].cpu().numpy(),
                "chi2": chi2.cpu().numpy()}
    logls = []
    for s in inputs:
        h, w = s["image"].shape
        step = max(1, 16_000_000 // (w * h))
        got = []
        for k in range(0, len(s["phys"]), step):
            m = _model(s["objects"], torch.tensor(s["phys"][k:k + step]), w, h, s["psf"], case["rule"])
            data, weight = torch.tensor(s["image"], device=m.device), torch.tensor(s["weight"], device=m.device)
            got.append(-0.5 * (weight.double() * (m - data.double()) ** 2).sum((1, 2)))
        logls.append(torch.cat(got).cpu().numpy())
    if case["entry"] == "systems":
        return {"logl": logls if len(logls) > 1 else logls[0]}
    # the physical parameters in sampler order: the free ones, then the fixed ones
    s = inputs[0]
    params = np.concatenate([s["phys"][:, s["free"]], s["phys"][:, ~s["free"]]], axis=1)
    if case["entry"] == "loglike":
        return {"logl": float(logls[0][0]), "params": params[0]}
    return {"logl": logls[0], "params": params}
