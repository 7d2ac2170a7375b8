"""The work this library's users have it do, as timed cases.

Each case is a dict of plain values; its "kind" names the entry point:

  tables     Engine.precompute of one or many parameter sets whose engine the
             program keeps: the captured graph of the batch is replayed
  changing   Engine.precompute where every call brings other parameters (an
             editor's sliders, a seasonal cycle): the plan is rebuilt per call
  host       precompute_host: one precompute into host arrays, what the drop-in
             preprocessAtmo does before it writes its files
  sky        consumer.sky_radiance, one ray per pixel
  aerial     consumer.in_scattering, one terrain point per pixel
  sunsky     consumer.sun_sky_irradiance, one (r, mu_s) pair per terrain vertex
  surrogate  Surrogate.precompute with the network trusted
  training   Surrogate.loss_grad, forward and backward of one training batch

Atmospheres are drawn around the batch distribution of the library (Rg, height,
scale heights, betas and the Mie g over the ranges of params.draw_set).  The
table consumer reads FP32 tables computed here (transmittance, single
scattering and the direct irradiance), so they do not depend on the library.

exact() evaluates the same passes in FP64 with plain torch.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "proland-4.0_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F8 = torch.float64
PI = 3.141592657            # the shaders' value of pi
EXACT_LOOKUPS = 4.0e9       # texel-directions up to which exact() covers a precompute


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _tables(name, kind, RR, RMU, RMUS, RNU, sets=1, mix=0, TW=256, TH=64, SW=64, SH=16, orders=4, NS=16, NI=32,
            IS=50, TS=500):
    c = dict(kind=kind, sets=sets, mix=mix, RR=RR, RMU=RMU, RMUS=RMUS, RNU=RNU, TW=TW, TH=TH, SW=SW, SH=SH,
             orders=orders, NS=NS, NI=NI, IS=IS, TS=TS)
    if name:
        c["name"] = name
    return c


def _consumer(name, kind, n, RR=32, RMU=128, RMUS=32, RNU=8, alt=0.2):
    c = dict(kind=kind, n=n, RR=RR, RMU=RMU, RMUS=RMUS, RNU=RNU, TW=256, TH=64, SW=64, SH=16, alt=alt)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest resolution class of the batch distribution: a preview table, launch latency counts
        _tables("preview_set", "tables", 16, 64, 16, 4),
        # the reference's default configuration
        _tables("earth_set", "tables", 32, 128, 32, 8),
        # the high-resolution precision study of bench.py
        _tables("precision_set", "tables", 64, 256, 64, 16, TW=512, TH=128, SW=128, SH=32, orders=8, NS=32),
        # sizes that fill no tile: odd columns, odd slices, other sample counts
        _tables("ragged_set", "tables", 21, 90, 27, 5, TW=200, TH=51, SW=50, SH=13, orders=3, NS=12, NI=20, IS=41,
                TS=333),
        # a catalogue of atmospheres in one batch, resolutions mixed from the three classes
        _tables("mixed_batch", "tables", 32, 128, 32, 8, sets=48, mix=1),
        # two states of an atmosphere editor: the engine sees new parameters on every call
        _tables("changing_set", "changing", 32, 128, 32, 8, sets=2),
        # the drop-in's precompute into host memory
        _tables("host_set", "host", 32, 128, 32, 8),
        # a full-HD sky from a camera near the ground
        _consumer("sky_frame", "sky", 1920 * 1080),
        # aerial perspective of a 720p view of the terrain
        _consumer("aerial_frame", "aerial", 1280 * 720, alt=3.0),
        # sun and sky light at the 65 x 65 vertices of a terrain tile
        _consumer("sun_tile", "sunsky", 65 * 65),
        # many unseen atmospheres at the reference resolution, orders >= 2 from the network
        _tables("surrogate_batch", "surrogate", 32, 128, 32, 8, sets=24),
        # one training batch of the study's size
        dict(name="training_batch", kind="training", n=65536),
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choice(["tables", "tables", "tables", "batch", "changing", "host", "sky", "aerial", "sunsky",
                       "surrogate", "training"])
    if kind in ("sky", "aerial", "sunsky"):
        return _consumer(None, kind, int(_log(rng, 500, 2.0e6)), RR=rng.randint(12, 48), RMU=2 * rng.randint(24, 96),
                         RMUS=rng.randint(8, 48), RNU=rng.randint(3, 12), alt=round(_log(rng, 0.05, 30.0), 3))
    if kind == "training":
        return dict(kind=kind, n=128 * int(_log(rng, 2, 512)))
    if kind == "batch":
        return _tables(None, "tables", 32, 128, 32, 8, sets=rng.randint(3, 40), mix=1, orders=rng.randint(2, 4),
                       NS=rng.choice([8, 12, 16]))
    if kind == "surrogate":
        return _tables(None, kind, rng.randint(12, 36), 2 * rng.randint(24, 70), rng.randint(10, 36),
                       rng.randint(4, 9), sets=rng.randint(1, 16))
    RR = int(_log(rng, 8, 64))
    RMU = 2 * int(_log(rng, 12, 128))
    RMUS = int(_log(rng, 6, 64))
    RNU = rng.randint(3, 16)
    small = kind in ("changing", "host")
    return _tables(None, kind, min(RR, 40) if small else RR, RMU, RMUS, min(RNU, 9) if small else RNU,
                   sets=2 if kind == "changing" else 1, TW=int(_log(rng, 48, 512)), TH=int(_log(rng, 16, 128)),
                   SW=int(_log(rng, 16, 128)), SH=rng.randint(6, 32), orders=rng.randint(2, 4 if small else 6),
                   NS=rng.randint(8, 16 if small else 32), NI=2 * rng.randint(6, 16), IS=rng.randint(24, 56),
                   TS=rng.randint(150, 500))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
CLASSES = ((16, 64, 16, 4), (32, 128, 32, 8), (48, 192, 48, 12))


def _f(x):
    return float(np.float32(x))


def _atmospheres(case, seed):
    """The case's parameter sets as dicts of FP32 values (held as floats)."""
    rng = random.Random(1000003 * seed + 17)
    out = []
    for i in range(case.get("sets", 1)):
        Rg = rng.uniform(3000.0, 7000.0)
        sR = rng.uniform(0.3, 3.0)
        bM = math.exp(rng.uniform(math.log(1e-3), math.log(3e-2)))
        a = dict(Rg=_f(Rg), Rt=_f(Rg + rng.uniform(40.0, 120.0)), HR=_f(rng.uniform(5.0, 12.0)),
                 HM=_f(rng.uniform(0.6, 2.4)), g=_f(rng.uniform(0.6, 0.9)), alpha=_f(0.1),
                 bR=[_f(b * sR) for b in (5.8e-3, 1.35e-2, 3.31e-2)], bMS=[_f(bM)] * 3, bME=[_f(bM / 0.9)] * 3)
        a["RL"] = _f(a["Rt"] + 1.0)
        RR, RMU, RMUS, RNU = CLASSES[i % 3] if case.get("mix") else (case["RR"], case["RMU"], case["RMUS"], case["RNU"])
        a.update(RR=RR, RMU=RMU, RMUS=RMUS, RNU=RNU, TW=case["TW"], TH=case["TH"], SW=case["SW"], SH=case["SH"])
        out.append(a)
    return out


def _params(a):
    from prolandatmo.params import earth
    return earth(Rg=a["Rg"], Rt=a["Rt"], RL=a["RL"], TRANSMITTANCE_W=a["TW"], TRANSMITTANCE_H=a["TH"], SKY_W=a["SW"],
                 SKY_H=a["SH"], RES_R=a["RR"], RES_MU=a["RMU"], RES_MU_S=a["RMUS"], RES_NU=a["RNU"],
                 AVERAGE_GROUND_REFLECTANCE=a["alpha"], HR=a["HR"], betaR=a["bR"], HM=a["HM"], betaMSca=a["bMS"],
                 betaMEx=a["bME"], mieG=a["g"])


def _options(case):
    from prolandatmo.params import options
    return options(orders=case["orders"], transmittance_samples=case["TS"], inscatter_samples=case["IS"],
                   irradiance_samples=case["NI"], spherical_samples=case["NS"])


def _buffers(atm):
    """One buffer per table kind, and each set's (T, E, S) views of it."""
    n, a0 = len(atm), atm[0]
    T = torch.zeros(n, a0["TH"], a0["TW"], 3, device=DEV)
    E = torch.zeros(n, a0["SH"], a0["SW"], 3, device=DEV)
    n4 = [a["RR"] * a["RMU"] * a["RMUS"] * a["RNU"] for a in atm]
    S = torch.zeros(sum(n4), 4, device=DEV)
    outs, o = [], 0
    for i, a in enumerate(atm):
        outs.append((T[i], E[i], S[o:o + n4[i]].view(a["RR"], a["RMU"], a["RNU"] * a["RMUS"], 4)))
        o += n4[i]
    return (T, E, S), outs


NIN, NH, NOUT, NHID = 14, 256, 4, 2
NORM = ((-9.0, -8.5, -8.0), (2.0, 2.0, 2.0), 1e-6)     # output standardisation (mu, sd, eps)


def _weights(seed):
    """Seeded FP32 parameter vector of the network (W1, b1, W2, b2, W3, b3, W5, b5)."""
    r = np.random.default_rng(seed + 71)
    parts = []
    for fin, fout in [(NIN, NH)] + [(NH, NH)] * NHID + [(NH, NOUT)]:
        a = math.sqrt(6.0 / (fin + fout))
        parts += [r.uniform(-a, a, fin * fout), r.uniform(-0.1, 0.1, fout)]
    return np.concatenate(parts).astype(np.float32)


def _batch(case, seed):
    """Rows as the training set holds them: coordinates and features in about [-2, 1.5], standardised targets."""
    g = torch.Generator(device="cpu").manual_seed(seed + 5)
    X = torch.rand(case["n"], 16, generator=g) * 2.0 - 1.0
    X[:, 14:] = 0.0
    T = torch.randn(case["n"], 4, generator=g)
    T[:, 3] = 0.0
    return X.to(DEV), T.to(DEV)


def _scene(case, seed):
    """FP32 tables of one atmosphere, the camera, the sun and the rays, points or vertices."""
    a = _atmospheres(case, seed)[0]
    c = dict(case, orders=1, IS=24, TS=200, NS=8, NI=8)
    T, E, S = _precompute64(a, c, direct_irradiance=True)
    T, E, S = (t.to(torch.float32).contiguous() for t in (T, E, S))
    rng = random.Random(seed + 29)
    cam = [0.0, 0.0, a["Rg"] + case["alt"]]
    az, el = rng.uniform(0, 2 * math.pi), rng.uniform(0.02, 1.2)
    sun = [math.cos(el) * math.cos(az), math.cos(el) * math.sin(az), math.sin(el)]
    n = case["n"]
    g = torch.Generator(device="cpu").manual_seed(seed + 3)
    if case["kind"] == "sunsky":
        h = torch.rand(n, generator=g, dtype=F8) * min(8.0, 0.2 * (a["Rt"] - a["Rg"]))
        m = torch.rand(n, generator=g, dtype=F8) * 1.25 - 0.25
        rows = torch.stack([a["Rg"] + h, m], -1).to(torch.float32).to(DEV)
        return a, T, E, S, cam, sun, rows
    # pixels of a perspective view, pitched at the horizon (sky) or down to the ground (aerial)
    w = max(1, int(math.sqrt(n * 16.0 / 9.0)))
    i = torch.arange(n, dtype=F8)
    u = (torch.remainder(i, w) + 0.5) / w * 2.0 - 1.0
    v = 1.0 - (torch.floor(i / w) + 0.5) / math.ceil(n / w) * 2.0
    yaw = rng.uniform(0, 2 * math.pi)
    pitch = rng.uniform(0.1, 0.5) if case["kind"] == "sky" else rng.uniform(-0.45, -0.25)
    fx, fz = math.tan(0.6) * 16.0 / 9.0, math.tan(0.6)
    x, y, z = torch.ones_like(u), u * fx, v * fz
    x, z = x * math.cos(pitch) - z * math.sin(pitch), x * math.sin(pitch) + z * math.cos(pitch)
    x, y = x * math.cos(yaw) - y * math.sin(yaw), x * math.sin(yaw) + y * math.cos(yaw)
    d = torch.stack([x, y, z], -1)
    d = d / d.norm(dim=-1, keepdim=True)
    if case["kind"] == "aerial":
        # distance to a terrain between 0 and 1.5 km high, at most 80 km; above the horizon a far ridge
        hgt = 0.75 + 0.75 * torch.sin(7.0 * u + 1.0) * torch.cos(5.0 * v)
        R = a["Rg"] + torch.clamp(hgt, max=0.9 * case["alt"])
        rmu = cam[2] * d[:, 2]
        q = rmu * rmu - cam[2] ** 2 + R * R
        t = torch.where((q > 0) & (rmu < 0), -rmu - torch.sqrt(q.clamp(min=0)), torch.full_like(q, 80.0))
        t = t.clamp(0.05, 80.0)
        d = torch.tensor(cam, dtype=F8) + d * t[:, None]
    rows = torch.nn.functional.pad(d, (0, 1)).to(torch.float32).contiguous().to(DEV)
    return a, T, E, S, cam, sun, rows


def prepare(case, seed):
    kind = case["kind"]
    if kind == "training":
        from prolandatmo.surrogate import Surrogate
        X, T = _batch(case, seed)
        s = Surrogate(0, seed=1)
        s.set_params(_weights(seed))
        return dict(kind=kind, s=s, X=X, T=T)
    if kind in ("sky", "aerial", "sunsky"):
        from prolandatmo import consumer as C
        a, T, E, S, cam, sun, rows = _scene(case, seed)
        return dict(kind=kind, p=_params(a), T=T, E=E, S=S, view=C.view(cam, sun), rows=rows)
    atm = _atmospheres(case, seed)
    st = dict(kind=kind, sets=[_params(a) for a in atm], opts=_options(case))
    if kind == "host":
        return st
    st["out"], st["outs"] = _buffers(atm)
    if kind == "surrogate":
        from prolandatmo.surrogate import Surrogate
        st["s"] = Surrogate(0, seed=1)
        st["s"].set_params(_weights(seed))
        st["s"].set_norm(*NORM)
    else:
        from prolandatmo.lib import Engine
        st["eng"] = Engine(0)
    return st


def run(st):
    kind = st["kind"]
    if kind == "tables":
        st["eng"].precompute(st["sets"], st["opts"], outs=st["outs"])
        return st["out"]
    if kind == "changing":
        for p, o in zip(st["sets"], st["outs"]):
            st["eng"].precompute([p], st["opts"], outs=[o])
        return st["out"]
    if kind == "host":
        from prolandatmo.lib import precompute_host
        return precompute_host(st["sets"][0], st["opts"])
    if kind == "surrogate":
        st["s"].precompute(st["sets"], st["opts"], outs=st["outs"], judge_fraction=0.0)
        return st["out"]
    if kind == "training":
        loss, grad = st["s"].loss_grad(st["X"], st["T"])
        return {"loss": np.float32(loss), "grad": grad}
    from prolandatmo import consumer as C
    if kind == "sky":
        return C.sky_radiance(st["p"], st["T"], st["S"], st["view"], st["rows"])
    if kind == "aerial":
        return C.in_scattering(st["p"], st["T"], st["S"], st["view"], st["rows"])
    return C.sun_sky_irradiance(st["p"], st["T"], st["E"], st["rows"])


def work(case):
    kind = case["kind"]
    if kind == "training":
        par = NIN * NH + NHID * NH * NH + NH * NOUT
        return {"bytes": case["n"] * (NIN + NOUT) * 4 + 2 * 4 * (par + 3 * NH + 4), "flops": 6 * par * case["n"]}
    if kind in ("sky", "aerial", "sunsky"):
        tab = (case["TW"] * case["TH"] * 3) * 4
        tab += case["SW"] * case["SH"] * 12 if kind == "sunsky" else case["RR"] * case["RMU"] * case["RMUS"] * case["RNU"] * 16
        row = 8 if kind == "sunsky" else 16
        # rays and results once; the tables at most once (a view touches a part of them)
        return {"bytes": case["n"] * (row + 32) + min(tab, case["n"] * 256),
                "flops": case["n"] * {"sky": 400, "aerial": 800, "sunsky": 120}[kind]}
    b = f = 0
    for a in _atmospheres(case, 0):
        n4, nT, nE = a["RR"] * a["RMU"] * a["RMUS"] * a["RNU"], a["TW"] * a["TH"], a["SW"] * a["SH"]
        b += n4 * 16 + (nT + nE) * 12
        f += nT * case["TS"] * 15 + n4 * (case["IS"] + 1) * 60
        if kind == "surrogate":
            f += (n4 + nE) * 2 * (NIN * NH + NHID * NH * NH + NH * NOUT)
        else:
            # a direction: its position (4), a linear piece of rgb (6), the weighted sum (6); order 2 has two
            # tables and the phase functions of the lookup (20 more)
            n = case["orders"] - 1
            f += n4 * 2 * case["NS"] ** 2 * (16 * n + 20 * min(n, 1)) + nE * case["NI"] ** 2 * 20 * n
            f += n4 * (case["IS"] + 1) * n * 50
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# the same passes in 64 bits
# ---------------------------------------------------------------------------
def _ar(n):
    return torch.arange(n, dtype=F8, device=DEV)


def _axis(x, n):
    """GL LINEAR with CLAMP_TO_EDGE along one axis: both texels and the weight of the second."""
    x = x.clamp(-1.0, float(n))
    f = torch.floor(x)
    k = f.long()
    return k.clamp(0, n - 1), (k + 1).clamp(0, n - 1), x - f


def _lookup2(tab, x, y):
    H, W = tab.shape[:2]
    i0, i1, a = _axis(x, W)
    j0, j1, b = _axis(y, H)
    t = tab.reshape(H * W, -1)
    a, b = a[..., None], b[..., None]
    return ((t[j0 * W + i0] * (1 - a) + t[j0 * W + i1] * a) * (1 - b)
            + (t[j1 * W + i0] * (1 - a) + t[j1 * W + i1] * a) * b)


def _uv_T(a, r, mu):
    ur = torch.sqrt(((r - a["Rg"]) / (a["Rt"] - a["Rg"])).clamp(min=0.0))
    um = torch.atan((mu + 0.15) / 1.15 * math.tan(1.5)) / 1.5
    return um * a["TW"] - 0.5, ur * a["TH"] - 0.5


def _T(a, T, r, mu):
    return _lookup2(T, *_uv_T(a, r, mu))


def _log_T(a, tau, r, mu):
    """log of the bilinear lookup of exp(-tau), without underflow."""
    x, y = _uv_T(a, r, mu)
    H, W = tau.shape[:2]
    i0, i1, u = _axis(x, W)
    j0, j1, v = _axis(y, H)
    t = tau.reshape(H * W, 3)
    taps = [(j0 * W + i0, (1 - u) * (1 - v)), (j0 * W + i1, u * (1 - v)), (j1 * W + i0, (1 - u) * v), (j1 * W + i1, u * v)]
    m = None
    for idx, w in taps:
        d = torch.where(w[..., None] > 0, t[idx], torch.full_like(t[idx], math.inf))
        m = d if m is None else torch.minimum(m, d)
    s = 0
    for idx, w in taps:
        s = s + torch.where(w[..., None] > 0, w[..., None] * torch.exp(m - t[idx]), torch.zeros_like(m))
    return torch.log(s) - m


def _segment(a, tau, r, mu, r1, mu1):
    """Transmittance of the ray from (r, mu) to the point (r1, mu1) on it."""
    r, mu = r.expand_as(r1), mu.expand_as(mu1)
    up = mu > 0
    x = _log_T(a, tau, torch.where(up, r, r1), torch.where(up, mu, -mu1))
    y = _log_T(a, tau, torch.where(up, r1, r), torch.where(up, mu1, -mu))
    return torch.exp((x - y).clamp(max=0.0))


def _limit(a, r, mu):
    k = r * r * (mu * mu - 1.0)
    out = -r * mu + torch.sqrt(k + a["RL"] ** 2)
    d2 = k + a["Rg"] ** 2
    din = -r * mu - torch.sqrt(d2.clamp(min=0.0))
    return torch.where((d2 >= 0) & (din >= 0), torch.minimum(out, din), out)


def _layer(a, l):
    """Radius and the four ray lengths of a layer as the FP32 uniforms hold them."""
    f = np.float32
    RgRg = f(f(a["Rg"]) * f(a["Rg"]))
    dRR = f(f(f(a["Rt"]) * f(a["Rt"])) - RgRg)
    r = l / (a["RR"] - 1.0)
    r = math.sqrt(float(RgRg) + r * r * float(dRR)) + (0.01 if l == 0 else (-0.001 if l == a["RR"] - 1 else 0.0))
    rho = math.sqrt(r * r - float(RgRg))
    return _f(r), _f(a["Rt"] - r), _f(rho + math.sqrt(float(dRR))), _f(r - a["Rg"]), _f(rho)


def _texels(a, l):
    """r, mu [RMU], mu_s [RMUS], nu [RNU] of a layer's texels."""
    r, dmin, dmax, dminp, dmaxp = _layer(a, l)
    n = a["RMU"]
    half = n * 0.5
    y = _ar(n)
    d0 = ((1.0 - y / (half - 1.0)) * dmaxp).clamp(min=dminp).clamp(max=dmaxp * 0.999)
    m0 = (a["Rg"] ** 2 - r * r - d0 * d0) / (2.0 * r * d0)
    m0 = m0.clamp(max=-math.sqrt(1.0 - (a["Rg"] / r) ** 2) - 0.001)
    d1 = ((y - half) / (half - 1.0) * dmax).clamp(min=dmin).clamp(max=dmax * 0.999)
    m1 = (a["Rt"] ** 2 - r * r - d1 * d1) / (2.0 * r * d1)
    mu = torch.where(y < half, m0, m1)
    muS = torch.tan((2.0 * _ar(a["RMUS"]) / (a["RMUS"] - 1.0) - 1.0 + 0.26) * 1.1) / math.tan(1.26 * 1.1)
    nu = -1.0 + _ar(a["RNU"]) / (a["RNU"] - 1.0) * 2.0
    return r, mu, muS, nu


def _coords4(a, rho2, rmu, mus):
    """Texel coordinates (z, y, x inside a nu slice) of texture4D at r^2 - Rg^2, r mu and mu_s."""
    H = math.sqrt(a["Rt"] ** 2 - a["Rg"] ** 2)
    rho = torch.sqrt(rho2.clamp(min=0.0))
    delta = rmu * rmu - rho2
    ground = (rmu < 0) & (delta > 0)
    fg = -rho / (torch.sqrt(delta.clamp(min=0.0)) - rmu)
    fs = (torch.sqrt((delta + H * H).clamp(min=0.0)) - rmu) / (rho + H)
    n = a["RMU"]
    u = torch.where(ground, 0.5 - 0.5 / n + fg * (0.5 - 1.0 / n), 0.5 + 0.5 / n + fs * (0.5 - 1.0 / n))
    z = (0.5 / a["RR"] + rho / H * (1.0 - 1.0 / a["RR"])) * a["RR"] - 0.5
    m = a["RMUS"]
    us = 0.5 / m + (torch.atan(mus.clamp(min=-0.1975) * math.tan(1.26 * 1.1)) / 1.1 + 0.74) * 0.5 * (1.0 - 1.0 / m)
    return z, u * n - 0.5, us * m - 0.5


def _tri(tab, z, y, x):
    RR, RMU, W = tab.shape[:3]
    k0, k1, c = _axis(z, RR)
    j0, j1, b = _axis(y, RMU)
    i0, i1, u = _axis(x, W)
    t = tab.reshape(RR * RMU * W, -1)
    s = 0
    for k, wk in ((k0, 1 - c), (k1, c)):
        for j, wj in ((j0, 1 - b), (j1, b)):
            row, w = (k * RMU + j) * W, wk * wj
            s = s + t[row + i0] * (w * (1 - u))[..., None] + t[row + i1] * (w * u)[..., None]
    return s


def _texture4(a, tab, rho2, rmu, mus, nu):
    z, y, x = _coords4(a, rho2, rmu, mus)
    p = (nu + 1.0) / 2.0 * (a["RNU"] - 1.0)
    k = torch.round(p)
    p = torch.where((p - k).abs() < 1e-9, k, p)
    f = torch.floor(p)
    w = (p - f)[..., None]
    z, y, x, f = torch.broadcast_tensors(z, y, x, f)
    m = float(a["RMUS"])
    return _tri(tab, z, y, f * m + x) * (1 - w) + _tri(tab, z, y, (f + 1.0) * m + x) * w


def _phases(a, nu):
    g = a["g"]
    q = 1.0 + nu * nu
    return (3.0 / (16.0 * PI) * q,
            1.5 / (4.0 * PI) * (1.0 - g * g) / (2.0 + g * g) * q * (1.0 + g * g - 2.0 * g * nu) ** -1.5)


def _rgb(v):
    return torch.tensor(v, dtype=F8, device=DEV)


def _transmittance64(a, case):
    y, x = torch.meshgrid(_ar(a["TH"]), _ar(a["TW"]), indexing="ij")
    r = a["Rg"] + ((y + 0.5) / a["TH"]) ** 2 * (a["Rt"] - a["Rg"])
    mu = -0.15 + torch.tan(1.5 * (x + 0.5) / a["TW"]) / math.tan(1.5) * 1.15
    n = case["TS"]
    dx = _limit(a, r, mu) / n
    sR, sM = torch.zeros_like(r), torch.zeros_like(r)
    for k in range(n + 1):
        t = k * dx
        h = torch.sqrt(r * r + t * t + 2.0 * t * r * mu) - a["Rg"]
        w = 0.5 if k in (0, n) else 1.0
        sR += w * torch.exp(-h / a["HR"])
        sM += w * torch.exp(-h / a["HM"])
    below = mu < -torch.sqrt(1.0 - (a["Rg"] / r) ** 2)
    dR, dM = (torch.where(below, torch.full_like(r, 1e9), s * dx)[..., None] for s in (sR, sM))
    tau = dR * _rgb(a["bR"]) + dM * _rgb(a["bME"])
    return torch.exp(-tau), tau


def _single64(a, case, T, tau):
    """Rayleigh and Mie single scattering [RR, RMU, RNU*RMUS, 3] without phase functions."""
    n = case["IS"]
    oR, oM = [], []
    for l in range(a["RR"]):
        r, mu, muS, nu = _texels(a, l)
        r = torch.tensor(r, dtype=F8, device=DEV)
        dx = _limit(a, r, mu) / n
        sR = torch.zeros(a["RMU"], a["RNU"], a["RMUS"], 3, dtype=F8, device=DEV)
        sM = torch.zeros_like(sR)
        rho2 = r * r - a["Rg"] ** 2
        for i in range(n + 1):
            t = i * dx
            q = rho2 + t * (t + 2.0 * r * mu)
            ri = torch.sqrt(q + a["Rg"] ** 2)
            seg = _segment(a, tau, r, mu, ri, (r * mu + t) / ri) * (0.5 if i in (0, n) else 1.0)
            num = nu[None, :, None] * t[:, None, None] + muS[None, None, :] * r
            seen = (num >= 0) | (num * num <= q[:, None, None])
            rc = ri.clamp(min=a["Rg"])
            sun = _T(a, T, rc[:, None, None].expand_as(num), num / ri[:, None, None])
            ti = torch.where(seen[..., None], seg[:, None, None, :] * sun, torch.zeros_like(sun))
            sR += ti * torch.exp(-(rc - a["Rg"]) / a["HR"])[:, None, None, None]
            sM += ti * torch.exp(-(rc - a["Rg"]) / a["HM"])[:, None, None, None]
        d = dx[:, None, None, None]
        oR.append((sR * d * _rgb(a["bR"])).reshape(a["RMU"], -1, 3))
        oM.append((sM * d * _rgb(a["bMS"])).reshape(a["RMU"], -1, 3))
    return torch.stack(oR), torch.stack(oM)


def _source64(a, case, tau, dE, tab):
    """The scattered radiance dJ of every texel; tab has 6 channels (Rayleigh, Mie) for order 2, else 3."""
    NS, first = case["NS"], tab.shape[-1] == 6
    out = []
    for l in range(a["RR"]):
        r0, mu, muS, nu = _texels(a, l)
        r = min(max(r0, a["Rg"]), a["Rt"])
        rho2 = torch.tensor(r * r - a["Rg"] ** 2, dtype=F8, device=DEV)
        mu = mu.clamp(-1.0, 1.0)[:, None, None]
        ms = muS.clamp(-1.0, 1.0)[None, None, :]
        var = torch.sqrt(1.0 - mu * mu) * torch.sqrt(1.0 - ms * ms)
        nn = torch.minimum(torch.maximum(nu[None, :, None], ms * mu - var), ms * mu + var)
        vx = torch.sqrt(1.0 - mu * mu)
        sx = torch.where(vx == 0, torch.zeros_like(nn), (nn - ms * mu) / vx)
        sy = torch.sqrt((1.0 - sx * sx - ms * ms).clamp(min=0.0))
        eR, eM = math.exp(-(r - a["Rg"]) / a["HR"]), math.exp(-(r - a["Rg"]) / a["HM"])
        acc = torch.zeros(a["RMU"], a["RNU"], a["RMUS"], 3, dtype=F8, device=DEV)
        phi = (_ar(2 * NS) + 0.5) * (PI / NS)
        for it in range(NS):
            th = (it + 0.5) * (PI / NS)
            ct, sn = math.cos(th), math.sin(th)
            wx, wy = torch.cos(phi) * sn, torch.sin(phi) * sn
            nu1 = sx[..., None] * wx + sy[..., None] * wy + (ms * ct)[..., None]
            nu2 = vx[..., None] * wx + (mu * ct)[..., None]
            pR, pM = _phases(a, nu2)
            rmu = torch.tensor(r * ct, dtype=F8, device=DEV)
            z, y, x = _coords4(a, rho2, rmu, ms[0, 0])
            # the nu slices of this direction's table row, one column beyond each end (CLAMP_TO_EDGE)
            k = (_ar(a["RNU"] + 2) - 1.0)[:, None]
            V = _tri(tab, *torch.broadcast_tensors(z, y, k * a["RMUS"] + x[None, :])).transpose(0, 1)
            p = (nu1 + 1.0) / 2.0 * (a["RNU"] - 1.0)
            f = torch.floor(p).clamp(-1.0, a["RNU"] - 1.0)
            w = (p - f)[..., None]
            row = (torch.arange(a["RMUS"], device=DEV) * (a["RNU"] + 2))[None, None, :, None] + f.long() + 1
            Vf = V.reshape(-1, V.shape[-1])
            L = Vf[row] * (1 - w) + Vf[row + 1] * w
            if first:
                qR, qM = _phases(a, nu1)
                L = L[..., :3] * qR[..., None] + L[..., 3:] * qM[..., None]
            if ct < -math.sqrt(1.0 - (a["Rg"] / r) ** 2):
                dg = -r * ct - math.sqrt(r * r * (ct * ct - 1.0) + a["Rg"] ** 2)
                mug = -(r * ct + dg) / a["Rg"]
                s2 = a["Rg"] ** 2 + dg * dg + 2.0 * a["Rg"] * mug * dg
                r1 = math.sqrt(s2)
                one = lambda v: torch.tensor([v], dtype=F8, device=DEV)  # noqa: E731
                tg = _segment(a, tau, one(a["Rg"]), one(mug), one(r1), one((a["Rg"] * mug + dg) / r1))[0]
                mg = (r * ms[..., None] + dg * nu1) / a["Rg"]
                e = _lookup2(dE, (mg + 0.2) / 1.2 * a["SW"] - 0.5, torch.full_like(mg, -0.5))
                L = L + a["alpha"] / PI * tg * e
            wgt = _rgb(a["bR"]) * eR * pR[..., None] + _rgb(a["bMS"]) * eM * pM[..., None]
            acc += (L * wgt).sum(3) * ((PI / NS) ** 2 * sn)
        out.append(acc.reshape(a["RMU"], -1, 3))
    return torch.stack(out)


def _irradiance64(a, case, tab):
    NI, first = case["NI"], tab.shape[-1] == 6
    j, i = torch.meshgrid(_ar(a["SH"]), _ar(a["SW"]), indexing="ij")
    h = j / (a["SH"] - 1.0) * (a["Rt"] - a["Rg"])
    r, muS = a["Rg"] + h, -0.2 + i / (a["SW"] - 1.0) * 1.2
    rho2 = h * (2.0 * a["Rg"] + h)
    sx = torch.sqrt((1.0 - muS * muS).clamp(min=0.0))
    acc = torch.zeros(a["SH"], a["SW"], 3, dtype=F8, device=DEV)
    for it in range(NI // 2):
        th = (it + 0.5) * PI / NI
        phi = (_ar(2 * NI) + 0.5) * PI / NI
        wz = math.cos(th)
        nu = sx[..., None] * (torch.cos(phi) * math.sin(th)) + (muS * wz)[..., None]
        L = _texture4(a, tab, rho2[..., None], (r * wz)[..., None], muS[..., None], nu)
        if first:
            qR, qM = _phases(a, nu)
            L = L[..., :3] * qR[..., None] + L[..., 3:] * qM[..., None]
        acc += L.sum(2) * (wz * (PI / NI) ** 2 * math.sin(th))
    return acc


def _gather64(a, case, tau, dJ):
    n = case["IS"]
    out = []
    for l in range(a["RR"]):
        r, mu, muS, nu = _texels(a, l)
        r = torch.tensor(r, dtype=F8, device=DEV)
        dx = _limit(a, r, mu) / n
        rho2 = r * r - a["Rg"] ** 2
        acc = torch.zeros(a["RMU"], a["RNU"], a["RMUS"], 3, dtype=F8, device=DEV)
        for i in range(n + 1):
            t = i * dx
            q = rho2 + t * (t + 2.0 * r * mu)
            ri = torch.sqrt(q + a["Rg"] ** 2)
            seg = _segment(a, tau, r, mu, ri, (r * mu + t) / ri) * (0.5 if i in (0, n) else 1.0)
            mi = (nu[None, :, None] * t[:, None, None] + muS[None, None, :] * r) / ri[:, None, None]
            v = _texture4(a, dJ, q[:, None, None], (r * mu + t)[:, None, None], mi, nu[None, :, None])
            acc += v * seg[:, None, None, :]
        out.append((acc * dx[:, None, None, None]).reshape(a["RMU"], -1, 3))
    return torch.stack(out)


def _precompute64(a, case, direct_irradiance=False):
    T, tau = _transmittance64(a, case)
    j, i = torch.meshgrid(_ar(a["SH"]), _ar(a["SW"]), indexing="ij")
    muS = -0.2 + i / (a["SW"] - 1.0) * 1.2
    dE = _T(a, T, a["Rg"] + j / (a["SH"] - 1.0) * (a["Rt"] - a["Rg"]), muS) * muS.clamp(min=0.0)[..., None]
    R, M = _single64(a, case, T, tau)
    S = torch.cat([R, M[..., :1]], -1)
    E = dE if direct_irradiance else torch.zeros_like(dE)
    tab = torch.cat([R, M], -1)
    nu = -1.0 + (_ar(a["RNU"]) / (a["RNU"] - 1.0) * 2.0).repeat_interleave(a["RMUS"])
    pr = (3.0 / (16.0 * PI) * (1.0 + nu * nu))[:, None]
    for _ in range(2, case["orders"] + 1):
        J = _source64(a, case, tau, dE, tab)
        dE = _irradiance64(a, case, tab)
        E = E + dE
        tab = _gather64(a, case, tau, J)
        S[..., :3] += tab / pr
    return T, E, S


def _act(z):
    t = (z / 6.0 + 0.5).clamp(0.0, 1.0)
    return z * t * t * (3.0 - 2.0 * t)


def _layers(w):
    out, o = [], 0
    w = torch.from_numpy(w).to(DEV).to(F8)
    for fin, fout in [(NIN, NH)] + [(NH, NH)] * NHID + [(NH, NOUT)]:
        out += [w[o:o + fin * fout].view(fin, fout), w[o + fin * fout:o + fin * fout + fout]]
        o += fin * fout + fout
    return out


def _network(w, x):
    for k in range(0, len(w), 2):
        x = x @ w[k] + w[k + 1]
        if k + 2 < len(w):
            x = _act(x)
    return x


def _features(a, S, E):
    """Network rows of every texel of S, then of E."""
    RR, RMU, RMUS, RNU = a["RR"], a["RMU"], a["RMUS"], a["RNU"]
    fs = [(a["Rg"] - 5000.0) / 2000.0, ((a["Rt"] - a["Rg"]) - 80.0) / 40.0, (a["HR"] - 8.5) / 3.5,
          (a["bR"][0] / 5.8e-3 - 1.65) / 1.35, (a["HM"] - 1.5) / 0.9,
          (math.log(a["bMS"][0]) + 5.2072) / 1.7006, (a["g"] - 0.75) / 0.15]
    Rg2, H = a["Rg"] ** 2, math.sqrt(a["Rt"] ** 2 - a["Rg"] ** 2)
    lo, hi, gap = 1e-3, 2.0 * H, 0.25
    l, y = _ar(RR)[:, None], _ar(RMU)[None, :]
    r = torch.sqrt(Rg2 + (l / (RR - 1)) ** 2 * H * H)
    r = r + torch.where(l == 0, 0.01, torch.where(l == RR - 1, -0.001, 0.0)).to(F8)
    rho = torch.sqrt((r * r - Rg2).clamp(min=0.0))
    half = RMU // 2
    d0 = torch.minimum(torch.maximum((1.0 - y / (half - 1)) * rho, r - a["Rg"]), 0.999 * rho)
    d1 = torch.minimum(torch.maximum((y - half) / (half - 1) * (rho + H), a["Rt"] - r), 0.999 * (rho + H))
    t = (torch.log(torch.where(y < half, d0, d1) / lo) / math.log(hi / lo)).clamp(0.0, 1.0)
    fy = torch.where(y < half, -(1 - gap) * t - gap, (1 - gap) * t + gap)
    shape = (RR, RMU, RNU, RMUS)
    c = [(2.0 * l / (RR - 1) - 1.0)[:, :, None, None].expand(shape), fy[:, :, None, None].expand(shape),
         (2.0 * _ar(RMUS) / (RMUS - 1) - 1.0).expand(shape),
         (2.0 * _ar(RNU) / (RNU - 1) - 1.0)[:, None].expand(shape)]
    n4 = RR * RMU * RNU * RMUS
    X = torch.stack([v.reshape(n4) for v in c], -1)
    j, i = torch.meshgrid(_ar(a["SH"]), _ar(a["SW"]), indexing="ij")
    two = torch.full_like(i, -2.0)
    XE = torch.stack([2.0 * j / (a["SH"] - 1) - 1.0, two, 2.0 * i / (a["SW"] - 1) - 1.0, two], -1).reshape(-1, 4)
    X = torch.cat([X, XE])
    ex = torch.cat([S.reshape(-1, S.shape[-1])[:, :3], E.reshape(-1, 3)])
    return torch.cat([X, _rgb(fs).expand(len(X), 7), 0.25 * (torch.log(ex.clamp(min=0.0) + 1e-6) + 5.0)], -1)


def _exact_surrogate(case, seed):
    w = _layers(_weights(seed))
    mu, sd, eps = _rgb(NORM[0]), _rgb(NORM[1]), NORM[2]
    Ts, Es, Ss = [], [], []
    for a in _atmospheres(case, seed):
        T, E, S = _precompute64(a, dict(case, orders=1))
        X = _features(a, S, E)
        v = torch.cat([_network(w, x)[:, :3] for x in X.split(1 << 19)])
        v = (torch.exp(v * sd + mu) - eps).clamp(min=0.0)
        n4 = S.shape[0] * S.shape[1] * S.shape[2]
        S = S.reshape(-1, 4)
        S[:, :3] += v[:n4]
        Ts.append(T)
        Es.append(E + v[n4:].view_as(E))
        Ss.append(S)
    return torch.stack(Ts), torch.stack(Es), torch.cat(Ss)


def _exact_training(case, seed):
    X, T = (t.to(F8) for t in _batch(case, seed))
    w = [v.clone().requires_grad_(True) for v in _layers(_weights(seed))]
    loss = ((_network(w, X[:, :NIN]) - T) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach(), "grad": torch.cat([v.grad.reshape(-1) for v in w])}


def _exact_consumer(case, seed):
    a, T, E, S, cam, sun, rows = _scene(case, seed)
    T, E, S, rows = (t.to(F8) for t in (T, E, S, rows))
    Rg, Rt = a["Rg"], a["Rt"]
    pad = torch.nn.functional.pad
    if case["kind"] == "sunsky":
        r, m = rows[:, 0], rows[:, 1]
        s = torch.where((m < -torch.sqrt(1.0 - (Rg / r) ** 2))[:, None], torch.zeros(1, 3, dtype=F8, device=DEV), _T(a, T, r, m))
        e = _lookup2(E, (m + 0.2) / 1.2 * a["SW"] - 0.5, (r - Rg) / (Rt - Rg) * a["SH"] - 0.5)
        return pad(s * 100.0, (0, 1)), pad(e * 100.0, (0, 1))
    cam, sun = _rgb(cam), _rgb(sun)

    def tex(r, mu, muS, nu):
        return _texture4(a, S, r * r - Rg * Rg, r * mu, muS, nu)

    def ratio(ra, ma, rb, mb, up):
        x = _T(a, T, torch.where(up, ra, rb), torch.where(up, ma, -mb))
        y = _T(a, T, torch.where(up, rb, ra), torch.where(up, mb, -ma))
        return torch.fmin(x / y, torch.ones_like(x))

    def colour(s, nu):
        pR, pM = _phases(a, nu)
        mie = s[:, :3] * (s[:, 3:] / s[:, :1].clamp(min=1e-4)) * _rgb([1.0, a["bR"][0] / a["bR"][1], a["bR"][0] / a["bR"][2]])
        return pad((s[:, :3] * pR[:, None] + mie * pM[:, None]) * 100.0, (0, 1))

    # the cameras here are inside the atmosphere: no ray has to be moved to its top
    r = torch.sqrt((cam * cam).sum()).expand(len(rows))
    if case["kind"] == "sky":
        v = rows[:, :3]
        rmu, nu, muS = v @ cam, v @ sun, (cam @ sun) / r
        mu = rmu / r
        return colour(tex(r, mu, muS, nu), nu), pad(_T(a, T, r, mu), (0, 1))
    pt = rows[:, :3]
    v = pt - cam
    dist = v.norm(dim=-1)
    v = v / dist[:, None]
    rmu, nu, muS = v @ cam, v @ sun, (cam @ sun) / r
    mu = rmu / r
    f = torch.where(r < Rg + 0.6, (Rg + 0.6) / r, torch.ones_like(r))
    r, pt = r * f, pt * f[:, None]
    r1 = pt.norm(dim=-1)
    mu1, muS1 = (pt * v).sum(-1) / r1, (pt @ sun) / r1
    e = ratio(r, mu, r1, mu1, mu > 0)
    e4 = torch.cat([e, e[:, :1]], -1)

    def diff(m, rr, mm):
        return (tex(r, m, muS, nu) - tex(rr, mm, muS1, nu) * e4).clamp(min=0.0)

    eps = 0.004
    lim = -torch.sqrt(1.0 - (Rg / r) ** 2)
    ends = []
    for m in (lim - eps, lim + eps):
        rr = torch.sqrt(r * r + dist * dist + 2.0 * r * dist * m)
        ends.append(diff(m, rr, (r * m + dist) / rr))
    w = ((mu - lim + eps) / (2.0 * eps))[:, None]
    s = torch.where(((mu - lim).abs() < eps)[:, None], ends[0] * (1 - w) + ends[1] * w, diff(mu, r1, mu1))
    t = (muS / 0.02).clamp(0.0, 1.0)
    s = torch.cat([s[:, :3], s[:, 3:] * (t * t * (3.0 - 2.0 * t))[:, None]], -1)
    return colour(s, nu), pad(e, (0, 1))


def exact(case, seed):
    kind = case["kind"]
    if kind == "training":
        return _exact_training(case, seed)
    if kind in ("sky", "aerial", "sunsky"):
        return _exact_consumer(case, seed)
    if kind == "surrogate":
        return _exact_surrogate(case, seed)
    atm = _atmospheres(case, seed)
    n = sum(a["RR"] * a["RMU"] * a["RMUS"] * a["RNU"] for a in atm) * 2 * case["NS"] ** 2 * (case["orders"] - 1)
    if n > EXACT_LOOKUPS:
        return None
    tabs = [_precompute64(a, case) for a in atm]
    if kind == "host":
        return tuple(t.cpu().numpy() for t in tabs[0])
    return (torch.stack([t[0] for t in tabs]), torch.stack([t[1] for t in tabs]),
            torch.cat([t[2].reshape(-1, 4) for t in tabs]))
