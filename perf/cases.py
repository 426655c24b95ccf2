"""The work that programs using this package ask of it, as cases to time.

A case is one pass through a public entry point of qsm_amd on the inputs that
entry point meets in use: the resident TV/TGV solver (qsm_amd.pd.Solver), the
whole single-step call on host arrays (qsm_amd.sstgv), the FFT dipole
convolution, the ADMM inversions (tv, rts), background removal (sharp, vsharp)
and Laplacian unwrapping, in single and double precision, on full and on
brain-shaped masks, at sizes from a small block to a whole-head 256 x 256 x
176 volume.

Volumes are column-major (x fastest): a torch volume is a contiguous (nz, ny,
nx) tensor seen through permute(2, 1, 0).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qsm.m_amd"))

from qsm_amd import bgremove, dipole, pd, rts, tv, unwrap  # noqa: E402
from qsm_amd.sstgv import sstgv  # noqa: E402

LARGEST = 256 * 256 * 176  # voxels of the largest volume


# ---- the cases --------------------------------------------------------------

def _case(path, shape, dtype, mask="ellipsoid", **more):
    nx, ny, nz = shape
    return dict(path=path, nx=nx, ny=ny, nz=nz, dtype=dtype, mask=mask, **more)


def listed():
    return [
        # a block cut around a small structure: launches and latency count
        dict(_case("tgv", (64, 64, 44), "float32", iters=100), name="tgv_small_f32"),
        # one echo of a head scan inside its brain mask, odd extents as a
        # crop to the mask's box leaves them
        dict(_case("tgv", (201, 235, 157), "float32", iters=100), name="tgv_brain_f32"),
        # the whole-head volume of the benchmark, every voxel active
        dict(_case("tgv", (256, 256, 176), "float32", mask="box", iters=100),
             name="tgv_large_f32"),
        # the same in double, MATLAB's own class
        dict(_case("tgv", (256, 256, 176), "float64", mask="box", iters=100),
             name="tgv_large_f64"),
        # total variation instead of TGV, anisotropic voxels
        dict(_case("tv", (167, 181, 121), "float32", iters=100, hz=1.5), name="tv_odd_f32"),
        # the drop-in call on host arrays with its own crop, lapw, stopping
        # rule and uncrop
        dict(_case("sstgv", (128, 128, 80), "float64", iters=200), name="sstgv_host_f64"),
        # the forward model of a whole head, zero padded to twice its size
        dict(_case("dipole", (256, 256, 176), "float32", mask="box"), name="dipole_large_f32"),
        # the ADMM inversion with tv.m's defaults on the whole head
        dict(_case("tv_admm", (256, 256, 176), "float32"), name="tv_admm_f32"),
        # the two-step inversion in double on a mid-size volume, tilted B0
        dict(_case("rts", (180, 216, 130), "float64", tilt=15.0), name="rts_f64"),
        # V-SHARP with its default radii on a volume cropped to the brain
        dict(_case("vsharp", (197, 233, 154), "float32"), name="vsharp_f32"),
        # unwrapping of the whole volume
        dict(_case("unwrap", (256, 256, 176), "float32", mask="box"), name="unwrap_large_f32"),
        # unwrapping inside a brain mask, in double, at odd extents
        dict(_case("unwrap", (161, 189, 123), "float64", hz=1.2), name="unwrap_brain_f64"),
    ]


def _smooth(n, primes):
    for p in primes:
        while n % p == 0:
            n //= p
    return n == 1


def draw(rng):
    path = rng.choice(["tgv", "tgv", "tv", "sstgv", "dipole", "tv_admm", "rts", "sharp", "vsharp",
                       "unwrap"])
    dtype = rng.choice(["float32", "float32", "float64"])
    while True:
        # slices are fewer than rows and columns, as in the scans
        nx, ny = (int(round(math.exp(rng.uniform(math.log(48), math.log(288))))) for _ in "xy")
        nz = int(round(math.exp(rng.uniform(math.log(40), math.log(200)))))
        if path in ("tv_admm", "rts"):  # the unpadded transforms' lengths
            nx, ny, nz = (next(m for m in range(n, 0, -1) if _smooth(m, (2, 3, 5, 7, 11, 13)))
                          for n in (nx, ny, nz))
        if nx * ny * nz <= (LARGEST // 4 if path == "sstgv" else LARGEST):
            break
    c = _case(path, (nx, ny, nz), dtype, mask=rng.choice(["ellipsoid", "ellipsoid", "box"]),
              hz=rng.choice([1.0, 1.2, 1.5]), tilt=rng.choice([0.0, 15.0]))
    if path in ("tgv", "tv", "sstgv"):
        c["iters"] = rng.randrange(40, 100)
    return c


# ---- inputs -------------------------------------------------------------------

def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _vsz(case):
    return (1.0, 1.0, case.get("hz", 1.0))


def _bdir(case):
    t = math.radians(case.get("tilt", 0.0))
    return (0.0, -math.sin(t), math.cos(t))


def _dt(case):
    return torch.float32 if case["dtype"] == "float32" else torch.float64


def _coords(case, dev):
    """Centred voxel indices, as (nz, ny, nx) broadcastable axes x, y, z."""
    nx, ny, nz = _shape(case)
    x = torch.arange(nx, device=dev, dtype=torch.float64) - (nx - 1) / 2
    y = torch.arange(ny, device=dev, dtype=torch.float64) - (ny - 1) / 2
    z = torch.arange(nz, device=dev, dtype=torch.float64) - (nz - 1) / 2
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _mask(case, dev):
    x, y, z = _coords(case, dev)
    nx, ny, nz = _shape(case)
    if case["mask"] == "box":
        return torch.ones((nz, ny, nx), dtype=torch.bool, device=dev)
    # fills most of its volume, as a brain does; the background removal's
    # device forms take a volume cropped to the mask, which touches its faces
    a, b, c = (0.5,) * 3 if case["path"] in ("sharp", "vsharp") else (0.46, 0.47, 0.46)
    return (x / (a * nx)) ** 2 + (y / (b * ny)) ** 2 + (z / (c * nz)) ** 2 <= 1.0


def _field(case, seed, dev):
    """A local field: the dipole field of 24 random rotated ellipsoids plus
    1 % noise, float64 (nz, ny, nx)."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = _shape(case)
    x, y, z = _coords(case, dev)
    s = min(nx, ny, nz)
    chi = torch.zeros((nz, ny, nx), dtype=torch.float32, device=dev)
    for _ in range(24):
        c = rng.uniform(-0.4, 0.4, 3) * (nx, ny, nz)
        ax = rng.uniform(0.03, 0.15, 3) * s + 1.5
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        v = float(rng.uniform(-0.2, 0.2))
        d = [(a - float(b)).float() for a, b in zip((x, y, z), c)]
        r2 = 0
        for k in range(3):
            u = (float(q[0, k]) * d[0] + float(q[1, k]) * d[1] + float(q[2, k]) * d[2])
            r2 = r2 + (u / float(ax[k])) ** 2
        chi += v * (r2 <= 1.0)
    M = [1 << math.ceil(math.log2(1.2 * n)) for n in (nz, ny, nx)]
    f = torch.fft.rfftn(chi, s=M)
    f *= _dipole(M[::-1], _vsz(case), _bdir(case), dev)[..., :M[2] // 2 + 1]
    f = torch.fft.irfftn(f, s=M)[:nz, :ny, :nx].double()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    noise = torch.randn((nz, ny, nx), generator=g, device=dev, dtype=torch.float64)
    return f + 0.01 * f.std() * noise


def _dipole(M, vsz, bdir, dev):
    """D = 1/3 - (k.b)^2 / k^2 on the transform grid, D(0) = 0 (M: x, y, z)."""
    kx, ky, kz = (torch.fft.fftfreq(n, h, dtype=torch.float64, device=dev) for n, h in zip(M, vsz))
    # an even axis's Nyquist sample stands at -n/2, as ifftshift leaves it
    kx, ky, kz = kx[None, None, :], ky[None, :, None], kz[:, None, None]
    k2 = kx * kx + ky * ky + kz * kz
    kb = bdir[0] * kx + bdir[1] * ky + bdir[2] * kz
    D = 1.0 / 3.0 - kb * kb / k2
    D[0, 0, 0] = 0.0
    return D


def _wrapped(case, seed, dev):
    """A wrapped phase: a local field and a smooth background, several turns
    across the volume."""
    x, y, z = _coords(case, dev)
    nx, ny, nz = _shape(case)
    f = _field(case, seed, dev)
    p = 20.0 * f + 9.0 * (x / nx) + 14.0 * (y / ny) ** 2 - 11.0 * (z / nz) ** 2
    return torch.remainder(p + math.pi, 2 * math.pi) - math.pi


def _neg_lap(u, vsz):
    """-Laplacian on the interior, zero on the faces."""
    out = torch.zeros_like(u)
    c = u[1:-1, 1:-1, 1:-1]
    hx, hy, hz = (1.0 / h ** 2 for h in vsz)
    out[1:-1, 1:-1, 1:-1] = -(hx * (u[1:-1, 1:-1, 2:] - 2 * c + u[1:-1, 1:-1, :-2])
                              + hy * (u[1:-1, 2:, 1:-1] - 2 * c + u[1:-1, :-2, 1:-1])
                              + hz * (u[2:, 1:-1, 1:-1] - 2 * c + u[:-2, 1:-1, 1:-1]))
    return out


def _inputs(case, seed, dev):
    """The volume a path takes and its mask, as (nz, ny, nx) in the case's
    precision and bool."""
    m = _mask(case, dev)
    path = case["path"]
    if path in ("tgv", "tv"):
        v = _neg_lap(_field(case, seed, dev), _vsz(case))
    elif path == "sstgv":
        v = torch.remainder(12.0 * _field(case, seed, dev) + math.pi, 2 * math.pi) - math.pi
    elif path == "unwrap":
        v = _wrapped(case, seed, dev)
    elif path in ("sharp", "vsharp"):
        x, y, z = _coords(case, dev)
        n = max(_shape(case))
        v = (_field(case, seed, dev) + 0.8 * (x * x - y * y) / n ** 2 + 0.5 * z / n) * m
    else:
        v = _field(case, seed, dev) * m
    return v.to(_dt(case)).contiguous(), m


def _vol(t):
    return t.permute(2, 1, 0)


# ---- one pass -----------------------------------------------------------------

LAM, ALPHA, TOL = 1e-3, 2.0, 3e-4
SHARP_R, THR = 9.0, 0.05


def _radii(case):
    return bgremove.default_radii(_vsz(case))


def prepare(case, seed):
    dev = torch.device("cuda")
    v, m = _inputs(case, seed, dev)
    shape, vsz, path, dt = _shape(case), _vsz(case), case["path"], _dt(case)
    s = dict(case=case, v=_vol(v), m=_vol(m.to(torch.uint8)))
    if path == "sstgv":
        # as MATLAB hands them over: host arrays, column-major
        s["v"] = np.asfortranarray(s["v"].cpu().numpy())
        s["m"] = np.asfortranarray(s["m"].cpu().numpy() != 0)
        return s
    s["out"] = _vol(torch.empty_like(v))
    if path in ("tgv", "tv"):
        s["solver"] = pd.Solver(pd._lib.TGV if path == "tgv" else pd._lib.TV, case["dtype"], shape,
                                vsz, LAM, ALPHA)
        return s
    if path == "dipole":
        s["pad"] = tuple(n // 2 for n in shape)
        nb = dipole.work_bytes(dt, shape, s["pad"])
    elif path == "tv_admm":
        nb = tv.work_bytes(dt, shape)
    elif path == "rts":
        nb = rts.work_bytes(dt, shape)
    elif path == "sharp":
        nb = bgremove.work_bytes(dt, shape, vsz, SHARP_R)
    elif path == "vsharp":
        nb = bgremove.vsharp_work_bytes(dt, shape, vsz, float(_radii(case).max()))
    else:
        nb = unwrap.work_bytes(dt, shape)
        s["d2"] = _vol(torch.empty_like(v))
    if path in ("sharp", "vsharp"):
        s["mo"] = _vol(torch.empty_like(m, dtype=torch.uint8))
    s["work"] = torch.empty(nb, dtype=torch.uint8, device=dev)
    return s


def run(s):
    case = s["case"]
    path, vsz = case["path"], _vsz(case)
    if path == "sstgv":
        return sstgv(s["v"], s["m"], vsz, LAM, ALPHA, TOL, case["iters"], False)
    if path in ("tgv", "tv"):
        return s["solver"].load(s["v"], s["m"]).iterate(case["iters"], 0.0).chi(s["out"])
    if path == "dipole":
        return dipole.dipole_conv_dev(s["v"], vsz, _bdir(case), s["pad"], s["out"], s["work"])
    if path == "tv_admm":
        tv.tv_dev(s["v"], s["m"], vsz, _bdir(case), {"verbose": 0}, s["out"], s["work"])
        return s["out"]
    if path == "rts":
        rts.rts_dev(s["v"], s["m"], vsz, _bdir(case), {"verbose": 0}, s["out"], s["work"])
        return s["out"]
    if path == "sharp":
        bgremove.sharp_dev(s["v"], s["m"], vsz, SHARP_R, THR, s["out"], s["mo"], s["work"])
        return s["out"], s["mo"]
    if path == "vsharp":
        bgremove.vsharp_dev(s["v"], s["m"], vsz, _radii(case), THR, s["out"], s["mo"], s["work"])
        return s["out"], s["mo"]
    unwrap.unwrap_laplacian_dev(s["v"], s["m"], vsz, s["out"], s["d2"], s["work"])
    return s["out"], s["d2"]


# ---- what a pass cannot do without ----------------------------------------------

def _smooth_up(n):
    while not _smooth(n, (2, 3, 5, 7)):
        n += 1
    return n


def work(case):
    """Bytes: each input read once, each output written once.  Flops: the
    updates, transforms and sweeps of the method itself, counted on the
    voxels it runs on."""
    nx, ny, nz = _shape(case)
    n, s, path = nx * ny * nz, (4 if case["dtype"] == "float32" else 8), case["path"]
    inside = n if case["mask"] == "box" else n * 4.0 / 3.0 * math.pi * 0.46 * 0.47 * 0.46
    by = (2 * s + 1) * n

    def fft(lengths):  # one real transform
        m = math.prod(lengths)
        return 2.5 * m * math.log2(m)

    if path in ("tgv", "sstgv"):
        return dict(bytes=by, flops=175.0 * inside * case["iters"])
    if path == "tv":
        return dict(bytes=by, flops=75.0 * inside * case["iters"])
    if path == "dipole":
        return dict(bytes=2 * s * n, flops=2 * fft([_smooth_up(2 * (k // 2) + k) for k in (nx, ny, nz)]))
    if path in ("tv_admm", "rts"):  # about nine ADMM steps with the default rule
        return dict(bytes=by, flops=9 * (2 * fft((nx, ny, nz)) + 90.0 * n))
    if path in ("sharp", "vsharp"):
        r = [SHARP_R] if path == "sharp" else list(_radii(case))
        pad = math.ceil(max(r) / min(_vsz(case)))
        m = [_smooth_up(k + 2 * pad) for k in (nx, ny, nz)]
        # the ball, the field and the mask per radius, and the last deconvolution
        return dict(bytes=by + n, flops=(3 + 3 * len(r)) * fft(m))
    # unwrapping: about twelve steps of two V-cycles, eight sweeps each at
    # 10 flops a voxel on the finest level, 8/7 over the levels
    return dict(bytes=by + s * n, flops=12 * (2 * 8 * 10 * 8 / 7 + 30) * inside)


# ---- the same results in 64 bits, in plain torch ---------------------------------

def _star(u, w):
    """w[0] (u-x + u+x) + w[1] (y) + w[2] (z) - 2 sum(w) u with zero outside
    (every caller's u is zero on the faces)."""
    r = torch.roll
    return (w[0] * (r(u, 1, 2) + r(u, -1, 2)) + w[1] * (r(u, 1, 1) + r(u, -1, 1))
            + w[2] * (r(u, 1, 0) + r(u, -1, 0))) - 2.0 * sum(w) * u


def _primal_dual(f, m, vsz, tgv, iters, tol):
    """The primal-dual TV/TGV iteration in float64 on (nz, ny, nx) volumes."""
    h = vsz
    gn = 4.0 * sum(1.0 / a ** 2 for a in h)
    wn = 6.0 * (1.0 / h[0] ** 2 + 1.0 / h[1] ** 2 + 2.0 / h[2] ** 2) / 3.0
    tau = 1.0 / math.sqrt(gn * gn + wn * wn)
    sig = 1.0 / (tau * (gn * gn + wn * wn))
    inner = torch.zeros_like(m)
    inner[1:-1, 1:-1, 1:-1] = True
    P = m & inner
    D = P.clone()
    for ax in range(3):
        D &= torch.roll(m, 1, ax) & torch.roll(m, -1, ax)
    P, D = P.double(), D.double()
    lap = [1.0 / a ** 2 for a in h]
    wav = [-1.0 / (3.0 * h[0] ** 2), -1.0 / (3.0 * h[1] ** 2), 2.0 / (3.0 * h[2] ** 2)]
    fw = lambda u, a: torch.roll(u, -1, 2 - a) - u     # noqa: E731
    bw = lambda u, a: u - torch.roll(u, 1, 2 - a)      # noqa: E731
    a1, a0 = LAM, ALPHA * LAM
    z = torch.zeros_like(f)
    chi, eta, chib, etab, nu = z.clone(), z.clone(), z.clone(), z.clone(), z.clone()
    p = [z.clone() for _ in range(3)]
    w = [z.clone() for _ in range(3)]
    wb = [z.clone() for _ in range(3)]
    q = [z.clone() for _ in range(6)]
    for it in range(1, iters + 1):
        nu += D * sig * ((_star(etab, lap) - _star(chib, wav)) + f)
        if tgv:
            p = [p[a] + D * sig * (fw(chib, a) / h[a] - wb[a]) for a in range(3)]
        else:
            p = [p[a] + D * sig * (fw(chib, a) / h[a]) for a in range(3)]
        s = torch.clamp(torch.sqrt(p[0] ** 2 + p[1] ** 2 + p[2] ** 2) / a1, min=1.0)
        p = [c / s for c in p]
        if tgv:
            g = [[fw(wb[c], a) / h[a] for a in range(3)] for c in range(3)]
            e = (g[0][0], 0.5 * (g[1][0] + g[0][1]), 0.5 * (g[2][0] + g[0][2]), g[1][1],
                 0.5 * (g[2][1] + g[1][2]), g[2][2])
            q = [a + D * sig * b for a, b in zip(q, e)]
            s = torch.sqrt(q[0] ** 2 + q[3] ** 2 + q[5] ** 2
                           + 2.0 * (q[1] ** 2 + q[2] ** 2 + q[4] ** 2))
            s = torch.clamp(s / a0, min=1.0)
            q = [c / s for c in q]
        eta1 = P * (eta - tau * _star(nu, lap)) / (1.0 + tau)
        div = bw(p[0], 0) / h[0] + bw(p[1], 1) / h[1] + bw(p[2], 2) / h[2]
        chi1 = chi + P * tau * (div + _star(nu, wav))
        if tgv:
            # each component of the divergence of q is scaled by that
            # component's own voxel size
            dq = [(bw(q[0], 0) + bw(q[1], 1) + bw(q[2], 2)) / h[0],
                  (bw(q[1], 0) + bw(q[3], 1) + bw(q[4], 2)) / h[1],
                  (bw(q[2], 0) + bw(q[4], 1) + bw(q[5], 2)) / h[2]]
            w1 = [w[a] + P * tau * (p[a] + dq[a]) for a in range(3)]
            wb = [2.0 * n - o for n, o in zip(w1, w)]
            w = w1
        chib, etab = 2.0 * chi1 - chi, 2.0 * eta1 - eta
        if tol > 0 and it % 10 == 0:
            n1 = torch.linalg.norm(chi1 - chi) / torch.linalg.norm(chi1)
            n2 = torch.linalg.norm(eta1 - eta) / torch.linalg.norm(eta1)
            if float(n1) < tol and float(n2) < 2.0 * tol:
                return chi1
        chi, eta = chi1, eta1
    return chi


def _lapw(u, vsz):
    """Sum over the axes of 1/h^2 times the difference of the wrapped one-sided
    differences, on the interior; zero on the faces."""
    def wrap(d):
        t = torch.fmod(d + math.pi, 2 * math.pi)
        t = torch.where(t < 0, t + math.pi, t - math.pi)
        return torch.where(d.abs() > math.pi, t, d)

    out = torch.zeros_like(u)
    acc = 0
    for a in range(3):
        d = wrap(torch.diff(u, dim=2 - a))
        e = torch.diff(d, dim=2 - a)
        for b in range(3):
            if b != a:
                e = e.narrow(2 - b, 1, e.shape[2 - b] - 2)
        acc = acc + e / vsz[a] ** 2
    out[1:-1, 1:-1, 1:-1] = acc
    return out


def _crop(m, grow):
    """The mask's box grown by `grow` voxels, clamped to the volume."""
    sl = []
    for a in range(3):
        k = torch.nonzero(m.any(dim=tuple(b for b in range(3) if b != a))).flatten()
        sl.append(slice(max(int(k[0]) - grow, 0), min(int(k[-1]) + grow + 1, m.shape[a])))
    return tuple(sl)


def _admm(u, F, K, vsz, o):
    """The ADMM loop shared by tv and rts on (nz, ny, nx) volumes."""
    N = u.numel()
    dims = u.shape
    L = 0
    for a in range(3):
        n = dims[2 - a]
        c = torch.cos(2 * math.pi * torch.arange(n, device=u.device, dtype=torch.float64) / n)
        L = L + ((2.0 - 2.0 * c) / vsz[a] ** 2).reshape([-1 if d == 2 - a else 1 for d in range(3)])

    def inv(rho):
        iA = 1.0 / (K + rho * L)
        iA[~torch.isfinite(iA)] = 0
        return iA

    grad = lambda x: [(torch.roll(x, -1, 2 - a) - x) / vsz[a] for a in range(3)]  # noqa: E731
    adj = lambda r: -sum((r[a] - torch.roll(r[a], 1, 2 - a)) / vsz[a] for a in range(3))  # noqa: E731
    mag = lambda r: float(torch.sqrt(r[0] ** 2 + r[1] ** 2 + r[2] ** 2).sum())    # noqa: E731
    rho, iA = o["rho"], inv(o["rho"])
    l = [torch.zeros_like(u) for _ in range(3)]
    v = grad(u)
    nr, flag = mag(v), 0
    for _ in range(20):
        u = torch.fft.ifftn(iA * (F + torch.fft.fftn(adj([rho * a - b for a, b in zip(v, l)])))).real
        g = grad(u)
        g1 = [1.5 * a - 0.5 * b for a, b in zip(g, v)]
        old = v
        v = [torch.sign(r) * torch.clamp(r.abs() - 1.0 / rho, min=0.0)
             for r in (a + b / rho for a, b in zip(g1, l))]
        l = [b + rho * (a - c) for a, b, c in zip(g1, l, v)]
        last, nr = nr, mag([a - b for a, b in zip(g, v)])
        ns = float(torch.linalg.norm(rho * adj([a - b for a, b in zip(v, old)])))
        ep = math.sqrt(3 * N) * o["atol"] + 0.1 * max(mag(g), mag(v))
        ed = math.sqrt(N) * o["atol"] + 0.1 * float(torch.linalg.norm(rho * adj(l)))
        if nr < ep and ns < ed:
            break
        if nr > 1e2 * ns or (nr > 0.7 * last and flag < 3):
            rho = 3.0 * rho
            iA = inv(rho)
            if flag > 5:
                flag = 0
        elif nr < ns / 1e2:
            rho, flag = rho / 9.0, flag + 1
            iA = inv(rho)
    return u


def _lsmr_diag(d, b, steps):
    """Fong and Saunders' LSMR for the diagonal operator d, `steps` steps."""
    norm = lambda x: float(torch.linalg.norm(x))     # noqa: E731
    beta = norm(b)
    u = b / beta
    v = d * u
    alpha = norm(v)
    v = v / alpha
    zb, ab, rho, rb, cb, sb = alpha * beta, alpha, 1.0, 1.0, 1.0, 0.0
    h, hb, x = v.clone(), torch.zeros_like(v), torch.zeros_like(v)
    for _ in range(steps):
        u = d * v - alpha * u
        beta = norm(u)
        u = u / beta
        v = d * u - beta * v
        alpha = norm(v)
        v = v / alpha
        ro, rho = rho, math.hypot(ab, beta)
        c, s = ab / rho, beta / rho
        th, ab = s * alpha, c * alpha
        rbo, thb = rb, sb * rho
        rb = math.hypot(cb * rho, th)
        cb, sb = cb * rho / rb, th / rb
        z, zb = cb * zb, -sb * zb
        hb = h - (thb * rho / (ro * rbo)) * hb
        x = x + (z / (rho * rb)) * hb
        h = v - (th / rho) * h
    return x


def _ball(M, r, vsz, dev):
    """The transform of the normalised ball centred on the origin (M: x, y, z)."""
    x, y, z = (((torch.arange(n, device=dev, dtype=torch.float64) + n // 2) % n - n // 2) * h
               for n, h in zip(M, vsz))
    b = ((y[None, :, None] ** 2 + x[None, None, :] ** 2) + z[:, None, None] ** 2 <= r * r).double()
    return torch.fft.fftn(b / b.sum()).real


def _background(f, m, vsz, radii, thr, single):
    """SHARP (single) or V-SHARP of a cropped volume, padded."""
    sz = f.shape
    pad = math.ceil(max(radii) / min(vsz))
    M = [_smooth_up(n + 2 * pad) for n in sz]
    off = [(a - n) // 2 + ((a - n) & 1 & n) for a, n in zip(M, sz)]
    box = tuple(slice(o, o + n) for o, n in zip(off, sz))
    fp = torch.zeros(M, dtype=torch.float64, device=f.device)
    mp = torch.zeros_like(fp)
    fp[box], mp[box] = f, m.double()
    F, S = torch.fft.fftn(fp), torch.fft.fftn(mp)
    acc, prev, inv, masks = 0, 0, None, []
    for r in radii:
        H = _ball(M[::-1], r, vsz, f.device)
        e = (torch.fft.ifftn(H * S).real > 0.999).double()
        h = 1.0 - H
        if inv is None:
            inv = 1.0 / h
            inv[h.abs() < thr] = 0
        acc = acc + (e - prev) * torch.fft.ifftn(h * F).real
        prev = e
        masks.append(e)
    out = prev * torch.fft.ifftn(inv * torch.fft.fftn(acc)).real
    # the mask that V-SHARP returns is the first of its last pair of radii
    mo = masks[-1] if single or len(radii) % 2 else masks[-2]
    return out[box].contiguous(), mo[box].to(torch.uint8).contiguous()


def _poisson(f, m, vsz):
    """-Lap v = f on the mask, v = 0 off it and past the faces: conjugate
    gradients in float64 to a relative residual of 1e-12."""
    pad = lambda t: torch.nn.functional.pad(t, (1,) * 6)     # noqa: E731
    g, w = pad(m.double()), [1.0 / h ** 2 for h in vsz]
    r = g * pad(f)
    x, p = torch.zeros_like(r), r.clone()
    rr = torch.sum(r * r)
    stop = 1e-24 * float(rr)
    for it in range(20000):
        q = -g * _star(p, w)
        a = rr / torch.sum(p * q)
        x += a * p
        r -= a * q
        new = torch.sum(r * r)
        p = r + (new / rr) * p
        rr = new
        if it % 50 == 49 and float(rr) <= stop:
            break
    return x[1:-1, 1:-1, 1:-1]


def exact(case, seed):
    dev = torch.device("cuda")
    v, m = _inputs(case, seed, dev)
    v, vsz, path = v.double(), _vsz(case), case["path"]
    dims = tuple(v.shape)
    if path in ("tgv", "tv"):
        return _vol(_primal_dual(v, m, vsz, path == "tgv", case["iters"], 0.0))
    if path == "sstgv":
        sl = _crop(m, 2)
        x = torch.zeros_like(v)
        x[sl] = _primal_dual(-_lapw(v[sl], vsz), m[sl], vsz, True, case["iters"], TOL)
        return x.permute(2, 1, 0).cpu().numpy()
    if path == "dipole":
        M = [_smooth_up(2 * (n // 2) + n) for n in dims]
        off = [(a - n) // 2 + ((a - n) & 1 & n) for a, n in zip(M, dims)]
        box = tuple(slice(o, o + n) for o, n in zip(off, dims))
        u = torch.zeros(M, dtype=torch.float64, device=dev)
        u[box] = v
        return _vol(torch.fft.ifftn(_dipole(M[::-1], vsz, _bdir(case), dev)
                                    * torch.fft.fftn(u)).real[box])
    if path == "tv_admm":
        D = _dipole(dims[::-1], vsz, _bdir(case), dev)
        return _vol(m * _admm(v, 7.5e3 * D * torch.fft.fftn(v), 7.5e3 * D * D, vsz,
                              dict(rho=9.0, atol=1e-4)))
    if path == "rts":
        D = _dipole(dims[::-1], vsz, _bdir(case), dev)
        if case["dtype"] == "float32":  # the region is chosen in the class of the field
            W = 1e5 * (D.float().abs() > 0.15).double()
        else:
            W = 1e5 * (D.abs() > 0.15).double()
        x1 = m * torch.fft.ifftn(_lsmr_diag(D, torch.fft.fftn(v), 4)).real
        return _vol(m * _admm(x1, W * torch.fft.fftn(x1), W, vsz, dict(rho=10.0, atol=1e-2)))
    if path in ("sharp", "vsharp"):
        one = path == "sharp"
        fl, ml = _background(v, m, vsz, [SHARP_R] if one else list(_radii(case)), THR, one)
        return _vol(fl), _vol(ml)
    d2 = _lapw(v, vsz)
    return _vol(_poisson(-d2, m, vsz)), _vol(d2)


def tolerance(case):
    """About four times the largest distance from exact() seen over the
    listed cases and forty drawn ones, per path and precision: the same sums
    in another order, no more."""
    single = case["dtype"] == "float32"
    path = case["path"]
    if path in ("tgv", "tv", "sstgv"):
        return dict(rel=1.6e-6, max=2.4e-5) if single else dict(rel=3e-15, max=4e-14)
    if path == "dipole":
        return dict(rel=8e-7, max=8e-6) if single else dict(rel=2e-15, max=2e-14)
    if path in ("tv_admm", "rts"):
        return dict(rel=1.6e-6, max=3e-5) if single else dict(rel=5e-15, max=8e-14)
    if path in ("sharp", "vsharp"):  # the deconvolution divides by 0.05 and more
        return dict(rel=1.3e-5, max=8e-5) if single else dict(rel=4e-14, max=3e-13)
    # the Poisson solve amplifies the rounding of its right-hand side by the
    # square of the volume's extent (single), or stops at 1e-8 (double)
    return dict(rel=2.7e-4, max=7e-4) if single else dict(rel=8e-8, max=1.2e-6)
