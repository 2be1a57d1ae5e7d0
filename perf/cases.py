"""Performance cases: the calls a user of this package makes, timed through its public entry points.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what the caller holds before the call, on the GPU (host arrays for `host`)
    run(state)           one pass through the public entry point, and its outputs
    work(case)           bytes and operations one pass cannot do without
    exact(case, seed)    the same outputs in 64-bit arithmetic, with torch alone

Kinds: `job` (one image on the device), `host` (numpy arrays in and out), `tiles` (a large image in
overlapping tiles), `batch` (several images through the engine), `psf` (a Born-Wolf PSF) and `output`
(statistics and the 16-bit volume a writer stores).

Images are Poisson counts of blurred points and blobs on a constant background; PSFs are Born-Wolf at
65 nm pixels.  Both are made with torch alone from the seed, so that they do not depend on the package.
Iteration counts are the lower end of what is used (10-25; the configurations of workloads.py run 20-100):
an iteration costs the same at any count, while heavy-ball trajectories amplify rounding with every one.
"""
import math

import numpy as np
import torch

import deconwolf_amd as dw
from deconwolf_amd import output, psf_bw, tiling
from deconwolf_amd.serve import Engine

DEV = "cuda:0"
TILE, OVERLAP = 512, 48   # the tiling of workloads.py's large image
DX, DZ, NA, NI = 65.0, 200.0, 1.40, 1.515


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _job(name, shape, psf, iters, bq=2, method="shb", rule="fixed", kind="job", n=1):
    M, N, P = shape
    pM, pN, pP = psf
    return {"name": name, "kind": kind, "M": M, "N": N, "P": P, "pM": pM, "pN": pN, "pP": pP, "iters": iters,
            "bq": bq, "method": method, "rule": rule, "n": n}


def listed():
    return [
        # a crop around one cell (the size of the package's smoke run): launches and host work are all of it
        _job("crop_40x36x16", (40, 36, 16), (9, 9, 7), 10),
        # a small stack, workloads.py's c1
        _job("c1_128x128x32", (128, 128, 32), (127, 127, 63), 20),
        # deconwolf's default stopping rule (REL, 2 %) on an odd-sized stack
        _job("rel_301x257x23", (301, 257, 23), (61, 61, 31), 0, rule="rel"),
        # the other method, ragged sizes
        _job("rl_701x533x37", (701, 533, 37), (101, 101, 51), 20, method="rl"),
        # a full camera frame with the default borders, workloads.py's c2
        _job("c2_1024x1024x60", (1024, 1024, 60), (181, 181, 79), 15),
        # no border padding (--bq 0): the transform is the image's own size
        _job("bq0_512x512x64", (512, 512, 64), (101, 101, 51), 20, bq=0),
        # half the border padding (--bq 1): deconwolf's exact size, 1115 x 1115 x 100
        _job("bq1_1024x1024x60", (1024, 1024, 60), (181, 181, 79), 10, bq=1),
        # numpy arrays in and out, as the Python wrapper of deconwolf is called
        _job("host_512x512x40", (512, 512, 40), (181, 181, 79), 20, kind="host"),
        # an image larger than the tile size, its tiles through the engine
        _job("tiles_1000x700x30", (1000, 700, 30), (101, 101, 51), 10, kind="tiles"),
        # a well of small images served together
        _job("batch_8x256x256x20", (256, 256, 20), (101, 101, 39), 20, kind="batch", n=8),
        # the PSF of one wavelength, workloads.py's size
        {"name": "psf_181x181x79", "kind": "psf", "N": 181, "P": 79, "nm": 520.0},
        # a c2 result on its way to a 16-bit TIFF
        {"name": "output_1024x1024x60", "kind": "output", "M": 1024, "N": 1024, "P": 60},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd(v):
    return v | 1


def draw(rng):
    kind = rng.choice(["job"] * 7 + ["host", "tiles", "batch", "psf", "output"])
    if kind == "psf":
        return {"kind": kind, "N": _odd(_log(rng, 31, 179)), "P": _odd(_log(rng, 15, 77)),
                "nm": rng.choice([460.0, 520.0, 600.0, 690.0])}
    if kind == "output":
        return {"kind": kind, "M": _log(rng, 64, 1024), "N": _log(rng, 64, 1024), "P": _log(rng, 8, 60)}
    bq = 2 if kind != "job" else rng.choice([2, 2, 2, 1, 0])
    if kind == "tiles":
        M, N, P = _log(rng, 520, 1000), _log(rng, 300, 700), _log(rng, 14, 30)
    elif kind == "batch":
        M, N, P = _log(rng, 64, 256), _log(rng, 64, 256), _log(rng, 10, 20)
    else:
        M, N, P = _log(rng, 32, 1024), _log(rng, 32, 1024), _log(rng, 8, 60)
    # PSFs no larger than deconwolf leaves after its crop to 2 * size - 1
    pM = _odd(_log(rng, 9, min(181, 2 * min(M, N) - 1)) - 1)
    pP = _odd(_log(rng, 7, min(79, 2 * P - 1)) - 1)
    if bq == 0:
        pM, pP = min(pM, _odd(min(M, N) - 2)), min(pP, _odd(P - 2))
    c = _job("", (M, N, P), (pM, pM, pP), rng.choice([10, 15] if bq == 2 else [10]), bq=bq, kind=kind)
    if kind == "batch":
        c["n"] = rng.choice([2, 4, 8])
    if kind == "job":
        c["method"] = rng.choice(["shb", "shb", "shb", "rl"])
        if bq == 2 and c["method"] == "shb" and rng.random() < 0.3:
            c["rule"], c["iters"] = "rel", 0
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs (torch alone)
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _smooth(n, even=False):
    """Smallest 2,3,5-smooth length >= n."""
    while True:
        m = n
        for f in (2, 3, 5):
            while m % f == 0:
                m //= f
        if m == 1 and not (even and n % 2):
            return n
        n += 1


def _gauss01(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return torch.tensor(0.5 * (x + 1), device=DEV), torch.tensor(0.5 * w, device=DEV)


def _profile(r_nm, z_nm, nm):
    """|A(r, z)|^2 of the Born-Wolf integral, one row per plane (float64)."""
    k0 = 2 * math.pi / nm
    zmax = float(z_nm.abs().max())
    n = int(96 + 2.0 * (k0 * NA * float(r_nm.max()) + k0 * NA * NA * zmax / (2 * NI)) / math.pi)
    rho, w = _gauss01(n)
    phase = -k0 * NA * NA / (2 * NI) * z_nm[:, None] * (rho * rho)[None, :]
    J = torch.special.bessel_j0(k0 * NA * r_nm[:, None] * rho[None, :]) * (rho * w)[None, :]
    return (torch.cos(phase) @ J.T) ** 2 + (torch.sin(phase) @ J.T) ** 2


def _psf(pM, pN, pP, nm=520.0):
    """Born-Wolf intensity at the pixel centres (linear in a profile of 8 samples per pixel), sum 1."""
    y = torch.arange(pN, device=DEV, dtype=torch.float64) - (pN - 1) / 2
    x = torch.arange(pM, device=DEV, dtype=torch.float64) - (pM - 1) / 2
    z = (torch.arange(pP, device=DEV, dtype=torch.float64) - (pP - 1) / 2) * DZ
    r = torch.sqrt(x[None, :] ** 2 + y[:, None] ** 2) * 8
    rs = torch.arange(int(float(r.max())) + 2, device=DEV, dtype=torch.float64)
    pr = _profile(rs * DX / 8, z, nm)
    i = r.floor().long()
    f = r - i
    v = pr[:, i] * (1 - f) + pr[:, i + 1] * f
    return (v / v.sum()).float().contiguous()


def _image(shape, psf, g):
    """(P, N, M) Poisson counts: points and blobs of U(200, 4000) on background 100, blurred by the PSF."""
    P, N, M = shape
    V = torch.zeros(P * N * M, device=DEV)
    n = max(8, int(2e-4 * V.numel()))
    at = torch.randint(0, V.numel(), (n,), generator=g, device=DEV)
    V.index_add_(0, at, 200 + 3800 * torch.rand(n, generator=g, device=DEV))
    V = V.view(1, 1, P, N, M)
    k = torch.exp(-0.5 * (torch.arange(-4, 5, device=DEV) / 1.5) ** 2)
    half = torch.zeros_like(V)
    half[..., : M // 2] = V[..., : M // 2]   # blobs on one side, points on the other
    for ax in range(3):
        w = k.view([9 if a == ax else 1 for a in range(3)])[None, None]
        half = torch.nn.functional.conv3d(half, w, padding=[4 if a == ax else 0 for a in range(3)])
    V = (torch.where(torch.arange(M, device=DEV) < M // 2, half, 5 * V))[0, 0]
    full = [_smooth(a + b - 1) for a, b in zip(shape, psf.shape)]
    B = torch.fft.irfftn(torch.fft.rfftn(V, full) * torch.fft.rfftn(psf, full), full)
    c = [(b - 1) // 2 for b in psf.shape]
    B = B[c[0]:c[0] + P, c[1]:c[1] + N, c[2]:c[2] + M].clamp_min(0) + 100.0
    return torch.poisson(B, generator=g).float().contiguous()


def _opts(case):
    s = dw.DwOpts()   # deconwolf's defaults: REL 2 %, at most 250 iterations
    if case["rule"] == "fixed":
        s.iter_type, s.nIter = dw.ITER_FIXED, case["iters"]
    s.borderQuality = case["bq"]
    s.method = dw.METHOD_RL if case["method"] == "rl" else dw.METHOD_SHB
    return s


def _inputs(case, seed):
    """(images without offset, psf)."""
    g = _gen(seed)
    psf = _psf(case["pM"], case["pN"], case["pP"])
    return [_image((case["P"], case["N"], case["M"]), psf, g) for _ in range(case["n"])], psf


def prepare(case, seed):
    kind = case["kind"]
    if kind == "psf":
        # another seed is another wavelength nearby
        return {"case": case, "nm": case["nm"] + (int(seed) % 1000) * 0.01}
    if kind == "output":
        return {"case": case, "vol": _result((case["P"], case["N"], case["M"]), seed), "bg": 100.0}
    ims, psf = _inputs(case, seed)
    st = {"case": case}
    if kind == "host":
        st["im"], st["psf"] = ims[0].cpu().numpy(), psf.cpu().numpy()
    elif kind == "tiles":
        st["im"], st["psf"] = ims[0], psf.cpu().numpy()
        st["engine"] = Engine(hbm_budget_gb=8.0, max_active=16)
    elif kind == "batch":
        st["ims"], st["psf"] = [v + 5.0 for v in ims], psf
        st["engine"] = Engine(hbm_budget_gb=8.0, max_active=16)
    else:
        st["im"], st["psf"] = ims[0] + 5.0, psf
    return st


def _result(shape, seed):
    """A deconvolved volume as the writers get it: background level in most voxels, bright structure."""
    g = _gen(seed)
    v = torch.rand(shape, generator=g, device=DEV)
    return torch.where(v < 0.6, torch.full_like(v, 100.0), 100.0 + 9000.0 * (v - 0.6) ** 3)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "psf":
        return psf_bw.bw_psf_device(case["N"], case["P"], state["nm"], NA=NA, ni=NI, dx_nm=DX, dz_nm=DZ)
    if kind == "output":
        vmax, nbg = output.stats(state["vol"], state["bg"])
        u16 = output.to_u16(state["vol"], output.scaling_for_u16(vmax), output.U16_ROUND)
        return {"max": vmax, "nbg": nbg, "u16": u16.view(np.int16)}
    s = _opts(case)
    if kind == "job":
        f = dw.deconvolve_rl_hip_device if case["method"] == "rl" else dw.deconvolve_shb_hip_device
        out = f(state["im"], state["psf"], s)
        return {"out": out, "err": s.err_trace, "iterations": s.stats["iterations"]}
    if kind == "host":
        out = dw.deconvolve(state["im"], state["psf"], case["iters"], bq=case["bq"], opts=s)
        return {"out": out, "err": s.err_trace, "iterations": s.stats["iterations"]}
    if kind == "tiles":
        out, _tiles, opts = tiling.deconvolve_tiles(state["im"], state["psf"], s, TILE, OVERLAP,
                                                    engine=state["engine"])
        return {"out": out, "err": [o.err_trace for o in opts]}
    eng = state["engine"]
    for i, im in enumerate(state["ims"]):
        eng.submit(i, im, state["psf"], s)
    left = len(state["ims"])
    while left:
        left -= len(eng.step())
    got = [eng.result(i) for i in range(len(state["ims"]))]
    return {"out": [o for o, _ in got], "err": [t["err_trace"] for _, t in got]}


# ---------------------------------------------------------------------------
# the least a pass has to do
# ---------------------------------------------------------------------------
def _sizes(case, M, N, P):
    d, p = (M, N, P), (case["pM"], case["pN"], case["pP"])
    if case["bq"] == 2:
        return [a + b - 1 for a, b in zip(d, p)]
    if case["bq"] == 1:
        return [a + (b + 1) // 2 for a, b in zip(d, p)]
    return [max(a, b) for a, b in zip(d, p)]


def work(case):
    """Bytes: per iteration the state (x_{k-1}, x_{k-2} and, with borders, W read, x_k written; RL has no
    x_{k-2}), the image and twice the OTF read, and each of the four transforms' half spectrum written and read once between
    axes; the inputs and the output.  Operations: 2.5 n log2 n per real transform and the pointwise steps."""
    if case["kind"] == "psf":
        n = case["N"]
        planes = (case["P"] + 1) // 2
        radii = 17 * (0.75 * n)
        return {"bytes": 4.0 * n * n * case["P"], "flops": planes * (radii * 200 * 60 + n * n / 8 * 64 * 10 * 8)}
    if case["kind"] == "output":
        v = case["M"] * case["N"] * case["P"]
        return {"bytes": 4.0 * v + 2.0 * v, "flops": 6.0 * v}
    boxes = [(case["M"], case["N"], case["P"])] * case["n"]
    if case["kind"] == "tiles":
        boxes = [(t[1] - t[0] + 1, t[3] - t[2] + 1, case["P"]) for _c, t in _tiles(case["M"], case["N"])]
    iters = case["iters"] or 10   # REL stops after about ten
    by = fl = 0.0
    for M, N, P in boxes:
        w = _sizes(case, M, N, P)
        V, img = float(w[0]) * w[1] * w[2], float(M) * N * P
        half = 8.0 * (w[0] // 2 + 1) * w[1] * w[2]
        state = 4.0 * V * ((3 if case["method"] == "shb" else 2) + (1 if case["bq"] else 0))
        by += iters * (state + 4 * img + 2 * half + 8 * half) + 8 * img
        fl += iters * (4 * 2.5 * V * math.log2(V) + 40 * V)
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _loop64(im, psf, case):
    """deconwolf's SHB or RL loop in float64 (src/method_shb.c:77-424, src/method_rl.c:105-400); im with
    the offset added.  Border quality 2 may run at any padded size: the image region does not change."""
    P, N, M = im.shape
    ref = _sizes(case, M, N, P)[::-1]
    w = [_smooth(v, i == 2) for i, v in enumerate(ref)] if case["bq"] == 2 else ref
    g, k = im.double(), psf.double()
    bg = max(float(g.min()), float(np.float32(1e-2)))
    z = torch.zeros(w, dtype=torch.float64, device=DEV)
    z[:k.shape[0], :k.shape[1], :k.shape[2]] = k
    at = int(torch.argmax(z))
    mid = (at // (w[1] * w[2]), at // w[2] % w[1], at % w[2])
    K = torch.fft.rfftn(torch.roll(z, [-v for v in mid], (0, 1, 2)))
    del z
    box = (slice(0, P), slice(0, N), slice(0, M))
    W = None
    if case["bq"] > 0:
        one = torch.zeros(w, dtype=torch.float64, device=DEV)
        one[box] = 1
        W = torch.fft.irfftn(K.conj() * torch.fft.rfftn(one), w)
        W = torch.where(W > 0.01, 1 / W.clamp_min(1e-3), torch.zeros_like(W))
        del one
    x = torch.full(w, float(np.float32(float(g.sum()) / (float(ref[0]) * ref[1] * ref[2]))), dtype=torch.float64,
                   device=DEV)
    xp = x.clone()
    rl, errs = case["method"] == "rl", []
    rel = case["rule"] == "rel"
    while len(errs) < (250 if rel else case["iters"]):
        i = len(errs)
        if rel and i:
            last = errs[-2] if i > 1 else 2 * errs[-1] * 0.02
            if abs(errs[-1] - last) / errs[-1] < 0.02:
                break
        a = 0.0 if rl else min(max((i - 1.0) / (i + 2.0), 0.0), 1.0)
        p = x if rl else (x + a * (x - xp)).clamp_min(bg)
        y = torch.fft.irfftn(K * torch.fft.rfftn(p), w)[box]
        errs.append(float((g * torch.log(g / y) - (g - y)).mean()))
        r = torch.full(w, 1e-6 if rl else 0.0, dtype=torch.float64, device=DEV)
        r[box] = g / y
        new = torch.fft.irfftn(K.conj() * torch.fft.rfftn(r), w)
        del r, y
        new *= p
        if W is not None:
            new *= W
        xp, x = x, new.clamp_min_(bg)
    return (x if rl else xp)[box].clone(), np.array(errs)


def _division(n, size):
    """Sections of tiling.c: [start, end] of ceil(n / size) parts."""
    parts = -(-n // size)
    cut = [0] + [int(math.ceil(float(np.float32(np.float32(n) / np.float32(parts)) * np.float32(d))))
                 for d in range(1, parts)] + [n]
    return [(a, b - 1) for a, b in zip(cut[:-1], cut[1:])]


def _tiles(M, N):
    """(core box, grown box) of deconwolf's XY tiling, each x0 x1 y0 y1."""
    out = []
    for a, b in _division(M, TILE):
        for c, d in _division(N, TILE):
            out.append(((a, b, c, d), (max(0, a - OVERLAP), min(M - 1, b + OVERLAP),
                                       max(0, c - OVERLAP), min(N - 1, d + OVERLAP))))
    return out


def _ramp(a, b, c, d, n):
    x = torch.arange(n, device=DEV, dtype=torch.float64)
    w = torch.where(x < b, (x - a + 1) / (b - a + 1), torch.where(x > c, 1 - (x - c) / (d - c + 1), torch.ones_like(x)))
    return torch.where((x < a) | (x > d), torch.zeros_like(x), w)


def _psf64(case, nm):
    """dw_bw's PSF (src/dw_bwpsf.c:538-775): pixel means of the Lanczos-5 interpolation of the profile."""
    N, P = case["N"], case["P"]
    c = (N - 1) / 2
    radmax = int(round(math.sqrt(2 * (N - c) ** 2))) + 1
    rs = torch.arange((radmax + 1) * 17 + 2, device=DEV, dtype=torch.float64)
    z = torch.tensor([float(np.float32(DZ * (i - (P - 1) / 2))) for i in range(P)], device=DEV, dtype=torch.float64)
    pr = _profile(rs * DX / 17, z, nm)
    gx, gw = _gauss01(8)
    x = torch.arange(N, device=DEV, dtype=torch.float64) - c
    X = x[:, None] + (gx - 0.5)[None, :]                    # pixel, node
    out = torch.zeros((P, N, N), dtype=torch.float64, device=DEV)
    k = torch.arange(-4, 6, device=DEV)
    for b in range(8):
        for a in range(8):
            r = 17 * torch.sqrt(X[:, b][:, None] ** 2 + X[:, a][None, :] ** 2)
            i = r.floor().long()
            t = (r - i)[..., None] - k
            wt = torch.sinc(t) * torch.sinc(t / 5)
            at = (i[..., None] + k).abs()
            for q in range(10):
                out += (gw[b] * gw[a]) * wt[..., q] * pr[:, at[..., q]]
    inside = torch.sqrt(x[:, None] ** 2 + x[None, :] ** 2) < radmax
    return out * inside


def exact(case, seed):
    kind = case["kind"]
    if kind == "psf":
        return _psf64(case, case["nm"] + (int(seed) % 1000) * 0.01)
    if kind == "output":
        v = _result((case["P"], case["N"], case["M"]), seed)
        return {"max": float(v.max()), "nbg": None, "u16": None}
    ims, psf = _inputs(case, seed)
    if kind == "batch":
        got = [_loop64(v + 5.0, psf, case) for v in ims]
        return {"out": [o for o, _ in got], "err": [e for _, e in got]}
    if kind == "tiles":
        P, N, M = ims[0].shape
        out, wsum, errs = (torch.zeros((P, N, M), dtype=torch.float64, device=DEV),
                           torch.zeros((N, M), dtype=torch.float64, device=DEV), [])
        for c, t in _tiles(M, N):
            wt = torch.minimum(_ramp(t[2], c[2], c[3], t[3], N)[:, None], _ramp(t[0], c[0], c[1], t[1], M)[None, :])
            box = (slice(t[2], t[3] + 1), slice(t[0], t[1] + 1))
            v, e = _loop64((ims[0][(slice(None),) + box] + 5.0).contiguous(), psf, case)
            errs.append(e)
            out[(slice(None),) + box] += wt[box] * (v - 5.0).clamp_min(0)
            wsum += wt
        return {"out": out / wsum, "err": errs}
    v, e = _loop64(ims[0] + 5.0, psf, case)
    return {"out": v, "err": e, "iterations": None}
