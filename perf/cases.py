"""Performance cases of the T2mapSEcorr / T2partSEcorr path: what its users run, through the public entry points.

A case is one call (T2 mapping of a volume with the T2 parts of its distribution, or T2 parts alone) with the options
and sizes of real use: a region of interest picked by hand, one slice, slabs of several slices; each regularization;
a measured B1 map, a fixed flip angle or the flip-angle search; plain FP64 and mixed precision; device-resident and
host arrays. `listed()` holds fixed cases, `draw(rng)` draws one more from the same ranges.

Inputs are the seeded synthetic multi-echo volumes that the tests and bench.py use (an ellipsoid mask of decaying
multi-component signals with Rician noise).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), os.pardir, "decaes.jl_amd"))
import decaes_amd as dmi  # noqa: E402
from decaes_amd import device as dmi_device  # noqa: E402

MAP_KEYS = ("gdn", "ggm", "gva", "fnr", "snr", "alpha", "resnorm", "mu", "chi2factor")


def _case(name, shape, nTE, nT2, reg, angles=32, TE=10e-3, T2lo=10e-3, ncomp=3, mask=0.6, entry="device",
          precision="fp64", flip="search", refcon=180.0):
    return dict(name=name, entry=entry, X=shape[0], Y=shape[1], Z=shape[2], nTE=nTE, nT2=nT2, TE=TE, T2lo=T2lo, reg=reg,
                angles=angles, ncomp=ncomp, mask=mask, precision=precision, flip=flip, refcon=refcon)


def listed():
    return [
        # a region of interest marked by hand on one slice, refitted while the user waits
        _case("roi_chi2", (4, 4, 1), 32, 40, "chi2", mask=1.0),
        # a small region through the host-array call that scripts use (numpy in, numpy out)
        _case("roi_gcv_host", (8, 8, 1), 48, 40, "gcv", mask=1.0, entry="host"),
        # a cropped block, the size of a quick check of an option set (bench.py's 32x32x4 workload)
        _case("block_chi2", (32, 32, 4), 32, 40, "chi2", mask=1.0),
        # a cropped block of odd sizes with a measured B1 map, unregularized
        _case("block_none_b1", (37, 29, 3), 33, 37, "none", mask=0.8, flip="b1"),
        # a block of a longer train with non-180 refocusing and the discrepancy principle
        _case("block_mdp_refcon", (61, 47, 2), 64, 60, "mdp", mask=0.8, refcon=172.0),
        # several slices at a known flip angle (phantoms, body-coil scans)
        _case("slices_chi2_fixed", (128, 128, 4), 48, 40, "chi2", flip="fixed"),
        # one 240x240 slice of the 48-echo protocol: GCV, the FP64 drop-in call
        _case("slice_gcv", (240, 240, 1), 48, 40, "gcv"),
        # one slice of the 56-echo brain protocol: L-curve, 64 angles
        _case("slice_lcurve", (240, 240, 1), 56, 60, "lcurve", angles=64, TE=7.9e-3, T2lo=8e-3, ncomp=4),
        # a slab of the 56-echo protocol with the regularization of the MATLAB toolbox
        _case("slab_chi2", (240, 240, 4), 56, 60, "chi2", angles=64, TE=7.9e-3, T2lo=8e-3, ncomp=4),
        # a slab of the 48-echo protocol
        _case("slab_gcv", (240, 240, 6), 48, 40, "gcv"),
        # a slab of the 56-echo protocol in mixed precision, as bench.py runs its volume
        _case("slab_lcurve_mixed", (240, 240, 4), 56, 60, "lcurve", angles=64, TE=7.9e-3, T2lo=8e-3, ncomp=4,
              precision="mixed"),
        # the T2 parts of a whole stored volume, recomputed with other windows
        _case("volume_t2part", (240, 240, 113), 56, 60, "lcurve", TE=7.9e-3, T2lo=8e-3, entry="t2part"),
    ]


def draw(rng):
    """One more case: any entry and option of the listed ones; sizes over the whole range, most of them odd."""
    entry = rng.choice(("device", "device", "device", "device", "host", "t2part"))
    nT2 = rng.choice((40, 60, rng.randint(16, 64)))
    nTE = rng.choice((24, 32, 48, 56, rng.randint(16, 64), rng.randint(16, 124)))
    if entry == "t2part":
        V = int(round(math.exp(rng.uniform(math.log(1e3), math.log(6.5e6)))))
    else:
        V = int(round(math.exp(rng.uniform(math.log(4), math.log(2.3e5)))))
    Z = rng.randint(1, max(1, min(48, V // 16)))
    Y = rng.randint(1, max(1, int(math.sqrt(V / Z)) * 2))
    X = max(1, round(V / (Y * Z)))
    reg = rng.choice(("none", "chi2", "gcv", "lcurve", "mdp"))
    flip = rng.choice(("search", "search", "search", "b1", "fixed"))
    c = dict(entry=entry, X=X, Y=Y, Z=Z, nTE=nTE, nT2=nT2, TE=rng.choice((7e-3, 7.9e-3, 10e-3)), T2lo=rng.choice((8e-3, 10e-3)),
             reg=reg, angles=rng.choice((16, 32, 64)), ncomp=rng.choice((3, 4)), mask=1.0 if V < 4096 else round(rng.uniform(0.3, 0.9), 3),
             precision=rng.choice(("fp64", "fp64", "mixed")), flip=flip, refcon=rng.choice((180.0, 180.0, 165.0)))
    most = max(work(x)["flops"] for x in listed())
    while entry != "t2part" and work(c)["flops"] > 0.8 * most:  # no dearer than the largest listed case
        c["X"], c["Y"] = max(1, c["X"] // 2), max(1, c["Y"] * 2 // 3)
    return c


# ------------------------------------------------------------------------------------------------------------
# what a user's program has before the call, and the call
# ------------------------------------------------------------------------------------------------------------
def _options(c):
    kw = dict(MatrixSize=(c["X"], c["Y"], c["Z"]), nTE=c["nTE"], TE=c["TE"], nT2=c["nT2"], T2Range=(c["T2lo"], 2.0),
              Reg=c["reg"], nRefAngles=c["angles"], RefConAngle=c["refcon"], SaveRegParam=True, SaveResidualNorm=True,
              Silent=True, precision=c["precision"])
    if c["reg"] == "chi2":
        kw["Chi2Factor"] = 1.02
    if c["reg"] == "mdp":
        kw["NoiseLevel"] = 2e-3
    if c["flip"] == "fixed":
        kw["SetFlipAngle"] = 165.0
    o = dmi.T2mapOptions(**kw)
    return o, dmi.T2partOptions.from_t2map(o, SPWin=(c["T2lo"], 40e-3), MPWin=(40e-3, 2.0))


def _image(c, seed):
    img, _ = dmi.synth_mse((c["X"], c["Y"], c["Z"]), c["nTE"], c["TE"], ncomp=c["ncomp"], mask_fraction=c["mask"], seed=seed)
    return img


def _b1(c, seed):
    return np.asfortranarray(np.random.default_rng(seed).uniform(130.0, 180.0, (c["X"], c["Y"], c["Z"])))


def _dist(c, seed):
    """A stored distribution volume, (nT2, Z, Y, X): a short and a long T2 peak in each voxel, NaN outside the mask."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n, V = c["nT2"], c["X"] * c["Y"] * c["Z"]
    r = torch.rand((4, V), dtype=torch.float64, device="cuda", generator=g)
    inside = torch.rand((V,), dtype=torch.float64, device="cuda", generator=g) < c["mask"]
    d = torch.empty((n, V), dtype=torch.float64, device="cuda")
    for j in range(n):
        u = j / (n - 1)
        short = torch.clamp(1 - (u - 0.15 - 0.1 * r[0]).abs() / 0.08, min=0) * r[1] * 0.2
        d[j] = torch.where(inside, short + torch.clamp(1 - (u - 0.45 - 0.2 * r[2]).abs() / 0.1, min=0) * (0.5 + r[3]), math.nan)
    return d.reshape(n, c["Z"], c["Y"], c["X"])


def _device(a):
    """A Julia-ordered (X, Y, Z, k) array as the contiguous (k, Z, Y, X) tensor of the same bytes."""
    return torch.from_numpy(np.ascontiguousarray(a.T)).cuda()


def _parts_out(c):
    f = torch.full((4, c["Z"], c["Y"], c["X"]), math.nan, dtype=torch.float64, device="cuda")
    return {k: f[i] for i, k in enumerate(("sfr", "sgm", "mfr", "mgm"))}


def prepare(case, seed):
    o, po = _options(case)
    s = dict(entry=case["entry"], o=o, po=po, alpha=None)
    if case["entry"] == "t2part":
        return dict(s, dist=_dist(case, seed), part=_parts_out(case))
    img = _image(case, seed)
    b1 = _b1(case, seed) if case["flip"] == "b1" else None
    if case["entry"] == "host":
        return dict(s, img=img, alpha=b1)
    out = dmi_device.alloc_t2map_outputs(o)
    if b1 is not None:
        s["alpha"] = _device(b1)
        out["alpha"].copy_(s["alpha"])
    return dict(s, img=_device(img), out=out, part=_parts_out(case))


def run(state):
    s = state
    if s["entry"] == "t2part":
        dmi_device.t2part_device(s["dist"], s["po"], s["part"])
        return dict(part=s["part"])
    if s["entry"] == "host":
        maps, dist = dmi.T2mapSEcorr(s["img"], s["o"], alpha=s["alpha"])
        part = dmi.T2partSEcorr(dist, s["po"])
        return dict(maps={k: maps[k].T for k in MAP_KEYS}, dist=dist.T, part={k: v.T for k, v in part.items()})
    dmi_device.t2map_device(s["img"], s["o"], s["out"], s["alpha"])
    dmi_device.t2part_device(s["out"]["dist"], s["po"], s["part"])
    return dict(maps={k: s["out"][k] for k in MAP_KEYS}, dist=s["out"]["dist"], part=s["part"])


def work(case):
    """Bytes: the image and the B1 map in, the distribution, the maps and the parts out. Flops: the Lawson-Hanson solves
    a voxel needs (flip-angle search, final solve and the regularization search), each as Householder QR with the size of
    the active set that such a solve ends with, the EPG basis at its angle and, for GCV, the spectrum of the basis."""
    m, n = case["nTE"], case["nT2"]
    V = case["X"] * case["Y"] * case["Z"]
    if case["entry"] == "t2part":
        return dict(bytes=8.0 * V * (n + 4), flops=V * case["mask"] * 7.0 * n)

    def solve(k):
        return 4.0 * m * n + sum(6.0 * (m - p) * (n - p) + p * p + 8.0 * (m - p) for p in range(min(k, m, n)))

    plain, reg = solve(4), solve(n // 3)
    f = 8 * plain if case["flip"] == "search" else 0.0
    f += 13.0 * n * (m * m / 4 + m) if case["flip"] != "fixed" else 0.0
    f += {"none": plain, "chi2": plain + 8 * reg, "mdp": plain + 8 * reg, "gcv": plain + 18 * reg, "lcurve": plain + 26 * reg}[case["reg"]]
    if case["reg"] == "gcv":
        N = min(m, n)
        f += 2.0 * N * N * max(m, n) + 4.0 / 3 * N ** 3 + 60.0 * N * N
    bytes_ = 8.0 * V * (m + n + len(MAP_KEYS) + 4 + (1 if case["flip"] == "b1" else 0))
    return dict(bytes=bytes_, flops=f * V * case["mask"])


# ------------------------------------------------------------------------------------------------------------
# the same results in plain numpy, for small volumes
# ------------------------------------------------------------------------------------------------------------
def _parts_exact(c, dist):
    """T2 parts of dist (voxels, nT2): fractions and geometric means of the short and middle windows."""
    T2 = np.exp(np.linspace(math.log(c["T2lo"]), math.log(2.0), c["nT2"]))
    T2[0], T2[-1] = c["T2lo"], 2.0
    lg, short, middle = np.log(T2), (T2 >= c["T2lo"]) & (T2 <= 40e-3), (T2 >= 40e-3) & (T2 <= 2.0)
    r = {}
    with np.errstate(all="ignore"):
        total = dist.sum(axis=1)
        for a, b, w in (("sfr", "sgm", short), ("mfr", "mgm", middle)):
            s = dist[:, w].sum(axis=1)
            r[a] = np.where(total > 0, s / total, np.nan)
            r[b] = np.where(s > 0, np.exp((dist[:, w] * lg[w]).sum(axis=1) / s), np.nan)
    return r


def _epg(alpha, m, TE, T2, T1=1.0, dual=False):
    """Echo amplitudes (K, m, n) of a constant-flip train for angles alpha (K,) in degrees, by the full recursion over
    phase states with refocusing pulses of alpha; with dual, also their derivatives by alpha in degrees."""
    a = np.deg2rad(np.atleast_1d(np.asarray(alpha, dtype=np.float64)))[:, None, None]
    E1, E2 = math.exp(-TE / 2 / T1), np.exp(-TE / 2 / T2)[None, :, None]
    sn, cs, d = np.sin(a), np.cos(a), math.pi / 180
    c2, s2 = np.cos(a / 2) ** 2, np.sin(a / 2) ** 2
    mix = ((c2 * E2 ** 2, s2 * E2 ** 2, sn * E1 * E2), (s2 * E2 ** 2, c2 * E2 ** 2, -sn * E1 * E2),
           (-sn / 2 * E1 * E2, sn / 2 * E1 * E2, cs * E1 ** 2))
    h = sn / 2 * d
    dmix = ((-h * E2 ** 2, h * E2 ** 2, cs * d * E1 * E2), (h * E2 ** 2, -h * E2 ** 2, -cs * d * E1 * E2),
            (-cs / 2 * d * E1 * E2, cs / 2 * d * E1 * E2, -sn * d * E1 ** 2))
    K, n, S = a.shape[0], len(T2), m + 2
    x, dx = [np.zeros((K, n, S)) for _ in range(3)], [np.zeros((K, n, S)) for _ in range(3)]
    x[0][:, :, 0] = 1.0
    m0, dm0 = np.sin(a / 2)[:, :, 0], (np.cos(a / 2) * d / 2)[:, :, 0]
    out, dout = np.zeros((K, m, n)), np.zeros((K, m, n))
    for i in range(m):
        y = [r[0] * x[0] + r[1] * x[1] + r[2] * x[2] for r in mix]
        dy = [r[0] * dx[0] + r[1] * dx[1] + r[2] * dx[2] + q[0] * x[0] + q[1] * x[1] + q[2] * x[2] for r, q in zip(mix, dmix)]
        e, de = y[1][:, :, 0], dy[1][:, :, 0]
        out[:, i], dout[:, i] = np.abs(m0 * e), np.sign(m0 * e) * (dm0 * e + m0 * de)
        for v, w in ((x, y), (dx, dy)):
            v[0] = np.concatenate([w[1][:, :, :1], w[0][:, :, :-1]], axis=2)
            v[1] = np.concatenate([w[1][:, :, 1:], np.zeros((K, n, 1))], axis=2)
            v[2] = w[2]
    return (out, dout) if dual else out


def _nnls(A, b, mu=0.0):
    """argmin |A x - b|^2 + mu^2 |x|^2 over x >= 0 (Lawson-Hanson), and the squared residual norm |A x - b|^2."""
    n = A.shape[1]
    G, h = (np.vstack([A, mu * np.eye(n)]), np.concatenate([b, np.zeros(n)])) if mu else (A, b)
    x, on = np.zeros(n), np.zeros(n, dtype=bool)
    for _ in range(3 * n):
        w = np.where(on, -np.inf, G.T @ (h - G @ x))
        tried = w.copy()
        moved = False
        while True:
            j = int(np.argmax(tried))
            if not tried[j] > 1e-14 * np.linalg.norm(h):
                break
            on[j] = True
            z = np.zeros(n)
            z[on] = np.linalg.lstsq(G[:, on], h, rcond=None)[0]
            if z[j] > 0:
                moved = True
                break
            on[j], tried[j] = False, -np.inf
        if not moved:
            break
        while np.any(z[on] <= 0):
            q = on & (z <= 0)
            t = np.min(x[q] / (x[q] - z[q]))
            x = x + t * (z - x)
            on &= x > 1e-300
            on[q & (x <= 1e-14 * np.max(np.abs(x)))] = False
            x[~on] = 0.0
            z = np.zeros(n)
            z[on] = np.linalg.lstsq(G[:, on], h, rcond=None)[0]
        x = z
    r = A @ x - b
    return x, float(r @ r)


def _cubic_min(a, b, u0, u1, m0, m1):
    """Minimum of the cubic Hermite segment on [a, b] with values u and slopes m at its ends."""
    best = (a, u0) if u0 < u1 else (b, u1)
    c = np.polynomial.polynomial.Polynomial([u0, m0 * (b - a), 3 * (u1 - u0) - (2 * m0 + m1) * (b - a), 2 * (u0 - u1) + (m0 + m1) * (b - a)])
    for t in c.deriv().roots():
        if abs(t.imag) < 1e-12 and 0 < t.real < 1 and c(t.real) < best[1] and c.deriv(2)(t.real) > 0:
            best = (a + t.real * (b - a), c(t.real))
    return best


def _search(angles, bases, dbases, b, least):
    """Flip angle minimizing the cubic Hermite surrogate of the loss over the angle grid, refined by bisection."""
    seen, K = {}, len(angles)

    def put(k):
        if k not in seen and len(seen) < K:
            x, res = _nnls(bases[k], b)
            seen[k] = (res, 2 * float((dbases[k] @ x) @ (bases[k] @ x - b)))
        return len(seen) >= K

    def suggest():
        ks = sorted(seen)
        best = (angles[ks[0]], seen[ks[0]][0])
        for p, q in zip(ks, ks[1:]):
            t = _cubic_min(angles[p], angles[q], seen[p][0], seen[q][0], seen[p][1], seen[q][1])
            best = t if t[1] < best[1] else best
        return best[0]

    def first(lo, hi, level):
        put(lo)
        put(hi)
        if len(seen) < least and level > 1:
            first(lo, (lo + hi) // 2, level - 1)
            first((lo + hi) // 2, hi, level - 1)

    for level in range(1, least + 1):
        first(0, K - 1, level)
        if len(seen) >= least:
            break
    x = suggest()
    while True:
        lo, hi = 0, K - 1
        while True:
            mid = (lo + hi) // 2
            box = (lo, mid) if angles[lo] <= x <= angles[mid] else (mid, hi)
            if not (box[0] in seen and box[1] in seen) or box[1] - box[0] <= 1:
                break
            lo, hi = box
        for k in sorted(box, key=lambda k: (angles[k] - x) ** 2):
            if not (box[0] in seen and box[1] in seen):
                put(k)
        x = suggest()
        if len(seen) >= K or box[1] - box[0] <= 1:
            return x


def exact(case, seed):
    """All outputs of a small volume with no regularization or a given flip angle, the search and the unregularized solve
    of others. None where the value is no number of its own: the regularization searches stop at a tolerance (a
    thousandth of the chi2 excess, 1e-4 in log mu), so mu, and what depends on it, is whichever point of that interval
    the steps reach."""
    c = case
    if c["entry"] == "t2part":
        d = _dist(c, seed).reshape(c["nT2"], -1).T.cpu().numpy()
        return dict(part={k: v.reshape(c["Z"], c["Y"], c["X"]) for k, v in _parts_exact(c, d).items()})
    V = c["X"] * c["Y"] * c["Z"]
    if V > (256 if c["flip"] == "search" else 4096) or c["refcon"] != 180.0 or c["precision"] != "fp64":
        return None
    m, n = c["nTE"], c["nT2"]
    T2 = np.exp(np.linspace(math.log(c["T2lo"]), math.log(2.0), n))
    T2[0], T2[-1] = c["T2lo"], 2.0
    img = _image(c, seed).reshape(V, m, order="F")
    alpha = np.full(V, np.nan)
    dist = np.full((V, n), np.nan)
    maps = {k: np.full(V, np.nan) for k in MAP_KEYS}
    if c["flip"] == "b1":
        alpha[:] = _b1(c, seed).reshape(V, order="F")
    angles = np.linspace(50.0, 180.0, c["angles"])
    if c["flip"] == "search":
        bases, dbases = _epg(angles, m, c["TE"], T2, dual=True)
    for i in np.flatnonzero(img[:, 0] > 0):
        top = img[i].max()
        b = img[i] / top
        if c["flip"] == "fixed":
            alpha[i] = 165.0
        elif c["flip"] == "search":
            alpha[i] = _search(angles, bases, dbases, b, min(5, c["angles"]))
        if c["reg"] != "none":
            continue
        A = _epg(alpha[i], m, c["TE"], T2)[0]
        x = _nnls(A, b)[0] * top
        r = A @ x - img[i]
        lg = np.log(T2)
        dist[i] = x
        g = (x * lg).sum() / x.sum()
        for k, v in (("gdn", x.sum()), ("ggm", math.exp(g)), ("gva", math.expm1(((lg - g) ** 2 * x).sum() / x.sum())),
                     ("fnr", x.sum() / math.sqrt((r @ r) / (m - 1))), ("snr", top / r.std(ddof=1)),
                     ("resnorm", math.sqrt(r @ r)), ("mu", 0.0), ("chi2factor", 1.0)):
            maps[k][i] = v
    maps["alpha"] = alpha
    shape = (c["Z"], c["Y"], c["X"])
    if c["reg"] != "none":
        return dict(maps={k: v.reshape(shape) if k == "alpha" else None for k, v in maps.items()}, dist=None,
                    part={k: None for k in ("sfr", "sgm", "mfr", "mgm")})
    return dict(maps={k: v.reshape(shape) for k, v in maps.items()}, dist=dist.T.reshape(n, *shape),
                part={k: v.reshape(shape) for k, v in _parts_exact(c, dist).items()})
