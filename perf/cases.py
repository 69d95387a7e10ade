"""Performance cases of the library: the calls a user's program makes, over the range of sizes and
options they are made with.

Every case is one realization (or one ensemble of realizations) through the public Python binding:
initialize, execute, finalize, as a program that computes one random field does. Grids and point
lists run the spectral method (method 1) on the kernel the library chooses, unless the case names
one; `fim` cases run the Fourier integral method (method 0). `host` cases take the field in a host
array (scarf_execute, the reference's call), the others in device memory (scarf_execute_device).

`exact` gives the same outputs in 64 bits from numpy and torch alone. The harmonics are *defined* at
the library's `real` precision (the reference rounds every wavenumber to it, and a wavenumber's
rounding is worth 1e-4 of the field far from the origin), so the draw is restated with the C
library's functions of that precision; everything after the draw is FP64.
"""
from __future__ import annotations

import bisect
import ctypes
import math

import numpy as np
import torch  # before the package: library and torch then share one HIP runtime

import scarf3d_amd
from scarf3d_amd.workloads import ensemble_members, init_library, structured_cfg, unstructured_cfg

PI = 3.141592653589793
M = 2147483647  # modulus of the random stream


def _grid(name, n, nharm, **kw):
    """A case's plain values with the defaults filled in."""
    c = dict(name=name, kind="grid", lib="f", host=False, kernel="auto", n1=n[0], n2=n[1], n3=n[2], nharm=nharm,
             ds=20.0, acf=0, hurst=0.25, cl1=500.0, cl2=500.0, cl3=500.0, sigma=0.05, alpha=0.0, beta=0.0,
             gamma=0.0, rescale=0, npoi=0, mute=20.0, taper=500.0, pad=0, npts=0)
    c.update(kw)
    return c


def listed():
    return [
        # a small block such as a test or an interactive session asks for: launches and latency
        _grid("grid_smallest", (32, 28, 24), 500, ds=50.0, cl1=500.0, cl2=400.0, cl3=300.0),
        # FP64 field of the reference's double precision build
        _grid("grid_128_double", (128, 128, 128), 5000, lib="d", ds=50.0, cl1=2000.0, cl2=2000.0, cl3=2000.0),
        # a production model with every option: odd sizes, rotated axes, rescaled, tapered, the
        # default harmonic count, the field in the caller's array
        _grid("grid_ragged", (301, 257, 129), 10000, host=True, ds=25.0, hurst=0.3, cl1=1500.0, cl2=1000.0,
              cl3=600.0, alpha=30.0, beta=20.0, gamma=10.0, rescale=1, npoi=3, mute=100.0, taper=400.0),
        # a 2D section with a Gaussian spectrum
        _grid("grid_2d", (1001, 701, 1), 10000, host=True, ds=10.0, acf=1, cl1=600.0, cl2=400.0, cl3=0.0),
        # the configuration the headline metric is quoted on
        _grid("grid_512", (512, 512, 512), 20000, ds=20.0, hurst=0.1, cl1=5000.0, cl2=5000.0, cl3=5000.0),
        # a caller that picks its field kernel (set_kernel)
        _grid("grid_256_fp16", (256, 256, 256), 10000, kernel="mfma_f16x2", ds=20.0, hurst=0.2, cl1=1500.0,
              cl2=1500.0, cl3=1500.0),
        # the largest benchmark model: rescaled, tapered around 16 points of interest
        _grid("grid_large", (1024, 1024, 512), 50000, ds=20.0, hurst=0.2, cl1=6000.0, cl2=4000.0, cl3=1500.0,
              sigma=0.08, rescale=1, npoi=16),
        # the nodes of an unstructured mesh
        _grid("points_2m", (10000, 10000, 5000), 10000, kind="points", host=True, npts=2_000_000, ds=50.0, acf=1,
              cl1=3000.0, cl2=3000.0, cl3=1000.0, sigma=0.1),
        # a coarser mesh in the double precision build
        _grid("points_double", (8000, 6000, 4000), 5000, kind="points", lib="d", npts=200_000, ds=50.0, hurst=0.3,
              cl1=1200.0, cl2=1000.0, cl3=800.0, sigma=0.08),
        # a Monte Carlo set of small realizations of uneven shape in one call
        _grid("ensemble_16", (0, 0, 0), 0, kind="ensemble", npts=16),
        # the reference examples' Fourier integral case
        _grid("fim_500", (500, 500, 500), 0, kind="fim", ds=50.0, cl1=2000.0, cl2=2000.0, cl3=2000.0),
        # the same method, double precision, padded, rescaled and tapered, into the caller's array
        _grid("fim_padded_double", (181, 160, 121), 0, kind="fim", lib="d", host=True, ds=50.0, hurst=0.3, cl1=800.0,
              cl2=600.0, cl3=400.0, rescale=1, npoi=2, mute=100.0, taper=800.0, pad=1),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["grid"] * 6 + ["points"] * 2 + ["fim"] * 2 + ["ensemble"])
    if kind == "ensemble":
        c = _grid("", (0, 0, 0), 0, kind=kind, npts=rng.randint(2, 15), host=False)
        del c["name"]
        c["first"] = rng.randint(0, 48)
        return c
    ds = rng.choice([10.0, 20.0, 25.0, 50.0])
    double = rng.random() < 0.3
    flat = kind != "points" and rng.random() < 0.15
    most = 3e7 if double else 3e8 if kind == "grid" else 1.4e8
    while True:
        if flat:
            n = [int(_log(rng, 40, 1600)), int(_log(rng, 40, 1600)), 1]
        elif kind == "points":  # extent of the box in metres
            n = [int(ds * rng.uniform(60, 220)) for _ in range(3)]
        else:
            n = [int(_log(rng, 20, 800)) for _ in range(3)]
        npts = int(_log(rng, 2000, 1.5e6)) if kind == "points" else 0
        nharm = int(_log(rng, 250, 30000))
        points = npts if npts else n[0] * n[1] * n[2]
        if points <= most and points * nharm <= (5e10 if double else 5e12):
            break
    span = [v if kind == "points" else (v - 1) * ds for v in n]
    acf = int(rng.random() < 0.3)
    cl = [rng.uniform(max(2.5 * ds, 0.06 * s), max(3 * ds, (0.3 if acf else 0.5) * s)) if s > 0 else 0.0 for s in span]
    c = _grid("", n, nharm, kind=kind, lib="d" if double else "f", host=rng.random() < 0.4, npts=npts, ds=ds, acf=acf,
              hurst=rng.choice([0.1, 0.2, 0.3, 0.5]), cl1=round(cl[0], 1), cl2=round(cl[1], 1), cl3=round(cl[2], 1),
              sigma=rng.choice([0.03, 0.05, 0.1]), rescale=int(rng.random() < 0.3), pad=int(rng.random() < 0.3))
    if kind == "grid" and not flat and rng.random() < 0.3:
        c.update(alpha=float(rng.randint(-60, 60)), beta=float(rng.randint(-30, 30)), gamma=float(rng.randint(-30, 30)))
    if rng.random() < 0.25:
        c.update(npoi=rng.randint(1, 6), mute=4 * ds, taper=12 * ds)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
def _seed(seed):
    """The realization's seed (a C int) of a preparation seed."""
    return 1 + (int(seed) * 48271 + 11) % 1_000_000_007


def _real(case):
    return np.float32 if case["lib"] == "f" else np.float64


def _config(case, seed):
    """The configuration dict of scarf3d_amd.workloads."""
    real = _real(case)
    cl = (case["cl1"], case["cl2"], case["cl3"])
    nd = 3 if cl[2] > 0 else 2
    poi = None
    if case["npoi"]:
        ext = np.array([v if case["kind"] == "points" else (v - 1) * case["ds"] for v in
                        (case["n1"], case["n2"], case["n3"])])[:nd]
        poi = np.random.default_rng(seed).uniform(0, 1, (nd, case["npoi"])) * ext[:, None]
    extra = dict(poi=poi, mute=case["mute"], taper=case["taper"]) if poi is not None else {}
    if case["kind"] == "points":
        cfg = unstructured_cfg(npts=case["npts"], box=(case["n1"], case["n2"], case["n3"]), dh=case["ds"],
                               acf=case["acf"], cl=cl, sigma=case["sigma"], hurst=case["hurst"], nharm=case["nharm"],
                               seed=seed, real=real, nd=nd, rescale=case["rescale"], **extra)
        for a in "xyz":  # the caller's coordinate arrays are of the library's `real`
            cfg[a] = cfg[a].astype(real)
    else:
        cfg = structured_cfg(n=(case["n1"], case["n2"], case["n3"]), ds=case["ds"], acf=case["acf"], cl=cl,
                             sigma=case["sigma"], hurst=case["hurst"], nharm=max(1, case["nharm"]),
                             alpha=case["alpha"], beta=case["beta"], gamma=case["gamma"], rescale=case["rescale"],
                             real=real, **extra)
    if case["kind"] == "fim":
        cfg["method"], cfg["pad"] = 0, case["pad"]
    return cfg


def _members(case, seed):
    """Ensemble members: shapes and spectra of the benchmark ensemble, seeds of their own."""
    first = case.get("first", 0)
    out = [dict(m) for m in ensemble_members()[first:first + case["npts"]]]
    for q, m in enumerate(out):
        m["seed"] = _seed(seed * 64 + q)
    return out


def _points(cfg):
    if not cfg["structured"]:
        return len(cfg["x"])
    return int(np.prod([cfg["fe"][i] - cfg["fs"][i] + 1 for i in range(3)]))


def prepare(case, seed):
    lib = scarf3d_amd.load(case["lib"])
    torch_real = torch.float32 if case["lib"] == "f" else torch.float64
    if case["kind"] == "ensemble":
        members = _members(case, seed)
        fields = [torch.zeros(int(np.prod(m["fe"])), dtype=torch_real, device="cuda") for m in members]
        return dict(lib=lib, members=members, fields=fields)
    cfg = _config(case, seed)
    n = _points(cfg)
    field = np.zeros(n, dtype=_real(case)) if case["host"] else torch.zeros(n, dtype=torch_real, device="cuda")
    return dict(lib=lib, cfg=cfg, seed=_seed(seed), field=field, host=case["host"], kernel=case["kernel"])


def run(state):
    lib = state["lib"]
    if "members" in state:
        stats = lib.ensemble_execute(state["members"], [f.data_ptr() for f in state["fields"]])
        return dict(fields=state["fields"], stats=stats[:, :4].copy())
    init_library(lib, state["cfg"])
    lib.set_kernel(state["kernel"])
    field = state["field"]
    if state["host"]:
        _, stats = lib.execute(state["seed"], out=field)
    else:
        stats = lib.execute_device(state["seed"], field.data_ptr())
    error = lib.last_error()
    lib.finalize()
    if error:
        raise RuntimeError(error)
    # stats(5:8) are timings
    return dict(field=field, stats=stats[:4].copy())


def work(case):
    """The least a pass moves and computes. The sum of nharm plane waves is a nonuniform Fourier transform:
    the direct sum takes 4 operations per point and harmonic, a fast transform about 5 log2 of the
    grid that resolves the model per grid point, plus the work at the harmonics and the points."""
    size = 4 if case["lib"] == "f" else 8
    if case["kind"] == "ensemble":
        shapes = [m["fe"] for m in _members(case, 0)]
        harmonics = sum(m["nharm"] for m in _members(case, 0))
        points = sum(int(np.prod(s)) for s in shapes)
        flops = sum(5 * np.prod(s) * math.log2(np.prod(s)) for s in shapes) + 100 * harmonics
        return dict(bytes=size * points + 40 * harmonics, flops=float(flops))
    n = [case["n1"], case["n2"], case["n3"]]
    if case["kind"] == "points":
        modes = math.prod(v / case["ds"] for v in n)
        return dict(bytes=size * 4 * case["npts"] + 40 * case["nharm"],
                    flops=5 * modes * math.log2(modes) + 100.0 * (case["npts"] + case["nharm"]))
    points = math.prod(n)
    if case["kind"] == "fim" and case["pad"]:
        points = math.prod(v + 2 * round(case["cl%d" % (i + 1)] / case["ds"]) for i, v in enumerate(n))
    return dict(bytes=size * math.prod(n) + 40 * case["nharm"],
                flops=5.0 * points * math.log2(points) + 100 * case["nharm"])


# ---------------------------------------------------------------------------
# The outputs in 64 bits
_libm = ctypes.CDLL("libm.so.6")


def _c(name, real):
    """The C library's function at `real`, over an array."""
    f = getattr(_libm, name + ("f" if real is np.float32 else ""))
    t = ctypes.c_float if real is np.float32 else ctypes.c_double
    f.restype = t

    def call(*arrays):
        n = max(np.size(a) for a in arrays)
        f.argtypes = [t] * len(arrays)
        cols = [np.broadcast_to(np.asarray(a, dtype=real), (n,)).tolist() for a in arrays]
        return np.array([f(*v) for v in zip(*cols)], dtype=real)

    return call


_A = (1498809829, 1160990996)  # recursion r = a0 r' + a1 r'' mod M; output g^r mod M
_G = 123567893
_tables = {}


def _powers(device):
    if device not in _tables:
        lo = [1]
        for _ in range(65535):
            lo.append(lo[-1] * _G % M)
        step = lo[-1] * _G % M
        hi = [1]
        for _ in range(32767):
            hi.append(hi[-1] * step % M)
        _tables[device] = (torch.tensor(lo, device=device), torch.tensor(hi, device=device))
    return _tables[device]


def _stream(seed, start, count, device):
    """Values start .. start + count - 1 of the seed's random stream (multiple recursive generator with
    an exponentiated output), uniform in [0, 1) in FP64."""
    def mul(x, y):
        return [(x[0] * y[0] + x[1] * y[2]) % M, (x[0] * y[1] + x[1] * y[3]) % M,
                (x[2] * y[0] + x[3] * y[2]) % M, (x[2] * y[1] + x[3] * y[3]) % M]

    def power(n):
        p, b = [1, 0, 0, 1], [_A[0], _A[1], 1, 0]
        while n:
            if n & 1:
                p = mul(p, b)
            b = mul(b, b)
            n >>= 1
        return p

    p = power(start)
    r0, r1 = (p[0] * (seed % M) + p[1]) % M, (p[2] * (seed % M) + p[3]) % M
    r = torch.empty(count + 2, dtype=torch.int64, device=device)  # r[0], r[1]: the state before the first value
    r[0], r[1] = r1, r0
    have = 2
    while have < count + 2:  # r[q + s] = (A^s)_00 r[q] + (A^s)_01 r[q - 1]
        s = have - 1
        p = power(s)
        k = min(s, count + 2 - have)
        r[have:have + k] = (p[0] * r[1:1 + k] + p[1] * r[0:k]) % M
        have += k
    r = r[2:]
    lo, hi = _powers(device)
    out = (hi[r >> 16] * lo[r & 65535]) % M
    out[r == 0] = 0
    return out.double() / M


def _integral(nd, acf, nu, k0, k1):
    """Integral of u^(nd-1) psd(u) over [k0, k1] in log u (k0 = 0, k1 = inf: the whole line)."""
    a, b = math.log(k0) if k0 > 0 else -30.0, math.log(k1) if math.isfinite(k1) else (230.0 if acf == 0 else 4.0)
    x, w = np.polynomial.legendre.leggauss(40)
    panels = max(1, math.ceil(2 * (b - a)))
    edge = np.linspace(a, b, panels + 1)
    t = (edge[:-1, None] + edge[1:, None]) / 2 + (edge[1:, None] - edge[:-1, None]) / 2 * x
    w = (edge[1:, None] - edge[:-1, None]) / 2 * w
    log_psd = -nu * np.logaddexp(0.0, 2 * t) if acf == 0 else -0.25 * np.exp(np.minimum(2 * t, 20.0))
    return float((w * np.exp(nd * t + log_psd)).sum())


def _harmonics(cfg, seed, r, device):
    """{wx, wy, wz, phase, amp} in FP64 of the kept harmonics, and the field's scaling."""
    f32 = r is np.float32
    cl = [r(c) for c in cfg["cl"]]
    nd = 3 if cl[2] > 0 else 2
    span = [r(cfg["fc"][i]) - r(cfg["nc"][i]) for i in range(3)]
    pi = r(PI)
    kmin = r(2) * pi * max(cl[i] / span[i] for i in range(nd))
    kmax, kc = (pi / r(cfg[d]) * min(cl[:nd]) for d in ("dh", "ds"))
    nu = r(cfg["hurst"]) + r(nd) / r(2)
    cnst = r(1) / np.sqrt(pi) if cfg["acf"] == 1 and nd == 3 else r(1)
    deg = [r(cfg[a]) * pi / r(180) for a in ("alpha", "beta", "gamma")]
    ca, cb, cg = _c("cos", r)(deg)
    sa, sb, sg = _c("sin", r)(deg)
    mat = np.array([[ca * cb, ca * sb * sg - sa * cg, ca * sb * cg + sa * sg],
                    [sa * cb, sa * sb * sg + ca * cg, sa * sb * cg - ca * sg], [-sb, cb * sg, cb * cg]], dtype=r)
    half = [s / r(2) for s in span]
    bar = [half[q] - (mat[q, 0] * half[0] + mat[q, 1] * half[1] + mat[q, 2] * half[2]) for q in range(3)]
    acf, nharm = cfg["acf"], cfg["nharm"]
    band = r(_integral(nd, acf, float(nu), float(kmin), float(kmax)))
    whole = r(_integral(nd, acf, float(nu), 0.0, math.inf))
    scaling = r(cfg["sigma"]) / np.sqrt(r(nharm)) * np.sqrt(band / whole)

    tr = torch.float32 if f32 else torch.float64

    def radial(u0):
        return u0 * float(kmax - kmin) + float(kmin)

    def acceptance(u):  # at `real`, the functions in FP64 and rounded
        if acf == 0:
            psd = 1 / torch.pow((1 + u * u).double(), float(nu)).to(tr)
        else:
            psd = torch.exp(-(0.25 * (u * u)).double()).to(tr)
        ud = u.double()
        return ((ud * psd.double() * (ud if nd == 3 else 1)) * float(cnst)).to(tr)

    # the stream in blocks of pairs; a pair passes as a trial whatever came before it
    blocks, accepted, pairs = [], [], 0
    size = 1 << 16

    def extend():
        nonlocal pairs, size
        v = _stream(seed, 2 * pairs, 2 * size, device).to(tr).view(-1, 2)
        ok = v[:, 1] < acceptance(radial(v[:, 0].clone()))
        accepted.extend((torch.nonzero(ok).flatten() + pairs).tolist())
        blocks.append(v)
        pairs += size
        size = min(2 * size, 1 << 23)

    def pair(q):  # values of the pairs q (ascending), from the blocks
        v = torch.empty(len(q), 2, dtype=tr, device=device)
        qt, at = torch.tensor(q, device=device), 0
        for b in blocks:
            m = (qt >= at) & (qt < at + len(b))
            v[m] = b[qt[m] - at]
            at += len(b)
        return v.cpu().numpy()

    kept, pos, done = [], 0, 0
    above = {}
    while done < nharm:
        p = bisect.bisect_left(accepted, pos)
        while p >= len(accepted) or accepted[p] + 4 > pairs:
            known = len(accepted)
            extend()
            if float(kc) < float(kmax):  # trials whose harmonic is dropped
                fresh = accepted[known:]
                u = radial(torch.as_tensor(pair(fresh)[:, 0]))
                above.update((q, True) for q, x in zip(fresh, u.tolist()) if x > float(kc))
            p = bisect.bisect_left(accepted, pos)
        q = accepted[p]
        done += 1
        if q in above:
            pos = q + 2
        else:
            kept.append(q)
            pos = q + 4
    q = np.array(kept)
    t0, t1, t2, t3 = (pair((q + k).tolist()) for k in range(4))
    u = radial(t0[:, 0].astype(r)).astype(r) if not f32 else (t0[:, 0] * (kmax - kmin) + kmin).astype(r)
    phi = t1[:, 0] * r(2) * pi
    sp, cp = _c("sin", r)(phi), _c("cos", r)(phi)
    if nd == 3:
        theta = _c("acos", r)(r(1) - r(2) * t1[:, 1])
        st, ct = _c("sin", r)(theta), _c("cos", r)(theta)
        v = [u * sp * st / cl[0], u * cp * st / cl[1], u * ct / cl[2]]
    else:
        v = [u * cp / cl[0], u * sp / cl[1], np.zeros_like(u)]
    normal = lambda t: np.sqrt(-(r(2) * _c("log", r)(t[:, 0]))) * _c("cos", r)(r(2) * pi * t[:, 1])  # noqa: E731
    a, b = normal(t2).astype(np.float64), normal(t3).astype(np.float64)
    v = np.stack(v).astype(np.float64)
    w = mat.astype(np.float64).T @ v
    phase = np.array(bar, dtype=np.float64) @ v - np.arctan2(a, b)
    return [torch.tensor(x, device=device) for x in (*w, phase, np.hypot(a, b))], float(scaling)


def _sum_grid(cfg, h, device):
    """Sum of the plane waves on the grid, FP64: a real product of e^(i wx x) with e^(i (wy y + wz z))."""
    wx, wy, wz, phase, amp = h
    ax = [torch.arange(cfg["fs"][i] - 1, cfg["fe"][i], device=device).double() * cfg["ds"] for i in range(3)]
    tx, ty = wx[:, None] * ax[0], ax[1][:, None] * wy
    x = torch.cat([torch.cos(tx), -torch.sin(tx)])
    y = torch.complex(torch.cos(ty), torch.sin(ty))
    out = []
    for z in ax[2].tolist():
        g = y * torch.polar(amp, wz * z + phase)
        out.append(torch.cat([g.real, g.imag], dim=1) @ x)
    return torch.stack(out)  # z, y, x


def _sum_points(cfg, h, device):
    wx, wy, wz, phase, amp = h
    p = [torch.tensor(np.asarray(cfg[a], dtype=np.float64), device=device) for a in "xyz"]
    out = torch.empty(len(p[0]), dtype=torch.float64, device=device)
    step = max(1, int(2e8) // len(amp))
    for i in range(0, len(out), step):
        s = slice(i, i + step)
        t = p[0][s, None] * wx + p[1][s, None] * wy + p[2][s, None] * wz
        out[s] = torch.cos(t.add_(phase)) @ amp
    return out


def _finish(f, cfg, axes, sigma, info):
    """Statistics, rescale and the tapers of a field whose coordinates broadcast to its shape."""
    sd, mean = float(f.std()), float(f.mean())
    if cfg["rescale"] == 1:
        f = f * (sigma / sd) - mean
        sd, mean = sigma, 0.0
    return _taper(f, cfg, axes), np.array([*info, sd, mean])


def _taper(f, cfg, axes):
    if cfg.get("poi") is None:
        return f
    for p in np.asarray(cfg["poi"]).T:
        d = torch.sqrt(sum((a - float(v)) ** 2 for a, v in zip(axes, p)) + 0.0)
        t = ((d - cfg["mute"]) / cfg["taper"]).clamp(0.0, 1.0)
        f = f * torch.where(d <= cfg["mute"], torch.zeros_like(d), 0.5 - 0.5 * torch.cos(PI * t))
    return f


def _flags(cfg):
    nd = 3 if cfg["cl"][2] > 0 else 2
    span = [cfg["fc"][i] - cfg["nc"][i] for i in range(3)]
    return [float(any(2 * PI / span[i] >= 1 / cfg["cl"][i] for i in range(nd))),
            float(any(cfg["ds"] > cfg["cl"][i] / 2 for i in range(nd)))]


def _exact_srm(cfg, seed, r, device):
    cfg = dict(cfg)
    if cfg.get("poi") is not None:
        cfg["poi"] = np.asarray(cfg["poi"]).astype(r).astype(np.float64)
    h, scaling = _harmonics(cfg, seed, r, device)
    if cfg["structured"]:
        f = _sum_grid(cfg, h, device).mul_(scaling)
        z, y, x = (torch.arange(cfg["fs"][i] - 1, cfg["fe"][i], device=device).double() * cfg["ds"] for i in (2, 1, 0))
        nd = 3 if cfg["cl"][2] > 0 else 2
        axes = [x[None, None, :], y[None, :, None], z[:, None, None]][:nd]
    else:
        f = _sum_points(cfg, h, device).mul_(scaling)
        axes = [torch.tensor(np.asarray(cfg[a], dtype=np.float64), device=device) for a in "xyz"][:cfg["nd"]]
    f, stats = _finish(f, cfg, axes, cfg["sigma"], _flags(cfg))
    return f.flatten(), stats


def _exact_fim(cfg, seed, r, device):
    """Random phases on the internal grid, Hermitian planes, backward transform, nearest neighbour. The
    grid's size and the neighbour of each point are decided at `real`."""
    dh, ds, cl = r(cfg["dh"]), r(cfg["ds"]), [r(c) for c in cfg["cl"]]
    nd = 3 if cl[2] > 0 else 2
    nint = lambda v: math.floor(float(v) + 0.5)  # noqa: E731
    npts, off = [], []
    for i in range(3):
        lo, hi = r(cfg["nc"][i]), r(cfg["fc"][i])
        extra = nint(cl[i] / dh) if cfg["pad"] == 1 else 0
        n = nint((((hi + dh * r(0.5)) - lo) + dh * r(0.5)) / dh) + 1 + 2 * extra
        o = lo - (r(extra) + r(0.5)) * dh
        npts.append(1 if nd == 2 and i == 2 else n + n % 2)
        off.append(-o if nd == 2 and i == 2 else o)
    n1, n2, n3 = npts
    h = n1 // 2 + 1
    flags = [float(any(npts[i] <= nint(r(2) * r(PI) * cl[i] / dh) for i in range(nd))),
             float(any(dh > cl[i] / r(2) for i in range(nd)))]
    k2 = 0.0
    for i, (n, shape) in enumerate(((n1, (1, 1, -1)), (n2, (1, -1, 1)), (n3, (-1, 1, 1)))):
        m = torch.arange(n, device=device)
        m = torch.minimum(m, n - m).double()
        dk = float((r(2) * r(PI)) / (r(n) * dh))
        k2 = k2 + (m[:h] if i == 0 else m).mul(dk * float(cl[i])).square().view(shape)
    hurst, sigma = float(r(cfg["hurst"])), float(r(cfg["sigma"]))
    nu = hurst + nd / 2
    volume = math.prod(float(c) for c in cl[:nd]) * sigma ** 2 * PI ** (nd / 2)
    if cfg["acf"] == 0:
        amp = torch.sqrt(2.0 ** nd * math.gamma(nu) / math.gamma(hurst) * volume * (1 + k2) ** -nu)
    else:
        amp = torch.sqrt(volume * torch.exp(-0.25 * k2))
    del k2
    s = torch.empty(n3, n2, h, dtype=torch.complex128, device=device)
    for k in range(0, n3, 64):
        m = min(64, n3 - k)
        u = _stream(seed, n1 * n2 * k, n1 * n2 * m, device).view(m, n2, n1)[:, :, :h]
        u = u.float().double() if r is np.float32 else u
        s[k:k + m] = torch.polar(amp[k:k + m].contiguous(), 2 * PI * u)
    jn, kn = n2 // 2, n3 // 2
    for p in (0, n1 // 2):
        b = s[:, :, p].clone()
        b[0, 0] = 0 if p == 0 else b[0, 0].real.clone()
        for k, j in ((kn, jn), (kn, 0), (0, jn)):
            if (k, j) != (0, 0):
                b[k, j] = b[k, j].real.clone()
        q = b.clone()
        if n3 > 1:
            mirror = torch.roll(b.flip(1), 1, 1)  # j -> -j mod n2
            q[kn + 1:] = mirror[1:n3 - kn].flip(0).conj()
            q[kn, jn + 1:] = b[kn, 1:n2 - jn].flip(0).conj()
            q[0, jn + 1:] = b[0, jn + 1:].conj()  # in place, as one process of the reference leaves it
        else:
            q[0, jn + 1:] = b[0, 1:n2 - jn].flip(0).conj()
        s[:, :, p] = q
    s = torch.fft.ifft(torch.fft.ifft(s, dim=0, norm="forward"), dim=1, norm="forward")
    for p in (0, n1 // 2):
        s[:, :, p] = s[:, :, p].real.clone()
    f = torch.fft.irfft(s, n=n1, dim=2, norm="forward")
    del s
    f /= math.sqrt(float(n1) * n2 * n3 * float(dh) ** nd)
    axes = [torch.arange(n, device=device).double().mul(float(dh)).view(v) for n, v in
            ((n1, (1, 1, -1)), (n2, (1, -1, 1)), (n3, (-1, 1, 1)))]
    inner = dict(cfg)
    if cfg.get("poi") is not None:
        inner["poi"] = np.stack([r(v) - off[i] for i, v in enumerate(np.asarray(cfg["poi"]).astype(r))]).astype(np.float64)
        axes = axes[:nd]
    f, stats = _finish(f, inner, axes, sigma, flags)
    index = []
    for i in range(3):
        c = ((np.arange(cfg["fs"][i] - 1, cfg["fe"][i]).astype(r) * ds - off[i]) / dh + r(3)) - r(1)
        inside = (c >= r(1)) & (c < r(npts[i] + 1))
        n = np.floor(c.astype(np.float64) + 0.5).astype(np.int64) - 2  # 0-based; -1 is the halo
        inside &= (n >= 0) | (i == 2)
        index.append((torch.tensor(np.where(inside, n % npts[i], 0), device=device), torch.tensor(inside, device=device)))
    (ix, ox), (iy, oy), (iz, oz) = index
    f = f[iz][:, iy][:, :, ix] * (oz[:, None, None] & oy[None, :, None] & ox[None, None, :])
    return f.flatten(), stats


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    r = _real(case)
    if case["kind"] == "ensemble":
        fields, stats = [], []
        for m in _members(case, seed):
            cfg = structured_cfg(n=m["fe"], ds=m["ds"], acf=m["acf"], cl=m["cl"], sigma=m["sigma"], hurst=m["hurst"],
                                 nharm=m["nharm"], real=r)
            f, s = _exact_srm(cfg, m["seed"], r, device)
            fields.append(f)
            stats.append(s)
        return dict(fields=fields, stats=np.stack(stats))
    cfg = _config(case, seed)
    field, stats = (_exact_fim if case["kind"] == "fim" else _exact_srm)(cfg, _seed(seed), r, device)
    return dict(field=field, stats=stats)
