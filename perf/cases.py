"""Performance cases: the calls a CT reconstruction program makes, over the range
of sizes, storage types and beam styles it makes them at.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and handles a program has before the call
    run(state)          one pass through the public entry points
    work(case)          bytes and operations a pass cannot do without
    exact(case, seed)   the same outputs in 64-bit torch arithmetic

The scenes are ten seeded ellipsoids (gpu_amd.phantom.ellipsoid_params).
Measurements are their analytic line integrals with Poisson noise, so the
inputs do not depend on any projector.  All lengths are millimetres; source
and detector lie at 1000 and 500 mm from the axis.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import numpy as np
import torch

from gpu_amd.autograd import project, tv_eps
from gpu_amd.core import Context
from gpu_amd.geometry import Geometry
from gpu_amd.phantom import ellipsoid_params, rotation_zyz

DSO, DOD = 1000.0, -500.0
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
I0 = 1e5
EPS = 1e-8   # of TV_eps
DEVICE = "cuda"


# --------------------------------------------------------------------- cases
def _scan(kind, name, nx, ny, nz, vx, cols, rows, du, views, **kw):
    c = dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, vx=vx, cols=cols, rows=rows, du=du, dv=du, views=views,
             dtype="f32", style=0, sources=1, src_z0=0.0, src_dz=0.0)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest reconstruction in use: a 32^3 volume, view by view; a
        # sweep is some forty launches of a few microseconds each
        _scan("sart", "sart_32", 32, 32, 24, 1.0, 48, 32, 1.0, 12, subset=1, order="ascending", beta=1.0),
        # the 128^3 / 180-view SART workload: one sweep in interleaved
        # subsets of 20 views
        _scan("sart", "sart_128_subsets", 128, 128, 128, 1.0, 256, 256, 1.0, 180, subset=20, order="interleaved",
              beta=1.0),
        # the benchmark volume and detector, view by view (the reference's
        # order), a sparse-view sweep of 64 views in FP32
        _scan("sart", "sart_512", 512, 512, 512, 0.5, 1024, 1024, 0.4, 64, subset=1, order="ascending", beta=0.02),
        # multi-slice fan beam with a row per slice, the reference's CT_style 1
        _scan("sart", "sart_fan_512", 512, 512, 256, 0.5, 1024, 256, 0.4, 24, subset=1, order="ascending", beta=0.05,
              style=1, dv=0.5),
        # a whole outer iteration (sweep, TV-FGP(20), momentum) with FP16
        # storage on a volume whose sides are no multiples of a tile
        _scan("iteration", "iteration_f16", 500, 468, 391, 0.5, 1000, 830, 0.4, 32, subset=1, order="ascending",
              beta=0.03, dtype="f16", lam=1e-3, inner=20),
        # gradient of 0.5 |Ax - b|^2 on the autograd test size: 64^3, 90 views
        _scan("gradient", "gradient_64", 64, 64, 64, 1.0, 96, 96, 1.0, 90),
        # the same at the benchmark size for a mini-batch of 16 views
        _scan("gradient", "gradient_512", 512, 512, 512, 0.5, 1024, 1024, 0.4, 16),
        # the multi-source workload with its TV_eps term: BF16 volume, 48
        # sources, 2 views
        _scan("gradient", "gradient_multisource_bf16", 256, 256, 256, 0.75, 1024, 128, 0.5, 2, dtype="bf16",
              sources=48, src_z0=-70.5, src_dz=3.0, lam=1e-3),
        # the objective that a reconstruction logs after each iteration
        _scan("objective", "objective_401", 401, 389, 300, 0.6, 768, 600, 0.5, 48, lam=1e-3),
        # TV-FGP denoising of the benchmark volume
        dict(name="tv_fgp_512", kind="tv_fgp", nx=512, ny=512, nz=512, vx=0.5, dtype="f32", lam=1e-3, inner=20),
        # FDK with the Hann window at the benchmark size, 360 views; as many
        # slices as the detector covers from every view
        _scan("fdk", "fdk_512", 512, 512, 416, 0.5, 1024, 1024, 0.4, 360, window="hann"),
        # FDK of a panel whose width is no power of two, FP16 projections
        _scan("fdk", "fdk_ragged_f16", 301, 307, 187, 0.6, 720, 475, 0.45, 240, window="ramp", dtype="f16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sart", "sart", "sart", "iteration", "gradient", "gradient", "objective", "tv_fgp", "fdk",
                       "fdk"])
    nx = _log_int(rng, 24, 420)
    ny = max(8, int(nx * rng.uniform(0.85, 1.15)))
    nz = max(8, int(nx * rng.uniform(0.4, 1.1)))
    width = rng.uniform(80.0, 256.0)
    vx = round(width / nx, 4)
    if kind == "tv_fgp":
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, vx=vx, dtype=rng.choice(["f32", "f16", "bf16"]),
                    lam=rng.choice([3e-4, 1e-3, 3e-3]), inner=rng.randint(5, 20))
    cols = int(nx * rng.uniform(1.3, 2.1))
    du = round(1.62 * vx * max(nx, ny) / cols, 4)
    rows = max(8, int(1.55 * vx * nz / du * rng.uniform(0.8, 1.1)))
    views = _log_int(rng, 4, 40)
    # an odd detector has rays on its midlines: with an even grid they would
    # run in the planes between voxels, where a ray belongs to neither side
    if cols % 2:
        nx, ny = nx | 1, ny | 1
    if rows % 2:
        nz = nz | 1
    if kind == "sart":
        style = rng.choice([0, 0, 0, 1, 2])
        views = _log_int(rng, 4, 60)
        subset = rng.choice([1, 1, min(4, views), min(10, views)])
        c = _scan(kind, "", nx, ny, nz, vx, cols, rows, du, views, style=style, subset=subset,
                  order=rng.choice(["ascending", "interleaved"]), beta=round(0.2 * subset ** 0.5, 3),
                  dtype=rng.choice(["f32", "f32", "f16", "bf16"]))
        if style:
            c.update(rows=nz, dv=vx)
    elif kind == "iteration":
        c = _scan(kind, "", nx, ny, nz, vx, cols, rows, du, views, subset=rng.choice([1, min(4, views)]),
                  order="ascending", beta=0.1, dtype=rng.choice(["f32", "f16", "bf16"]), lam=1e-3,
                  inner=rng.randint(5, 20))
    elif kind == "gradient":
        ns = rng.choice([1, 1, rng.randint(2, 24)])
        c = _scan(kind, "", nx, ny, nz, vx, cols, rows, du, max(2, views // (2 if ns == 1 else ns)),
                  dtype=rng.choice(["f32", "f16", "bf16"]))
        if ns > 1:
            dz = round(rng.uniform(2.0, 4.0), 2)
            c.update(sources=ns, src_z0=-dz * (ns - 1) / 2.0, src_dz=dz, rows=max(8, rows // 4))
        if rng.random() < 0.5:
            c.update(lam=rng.choice([1e-3, 1e-1]))
    elif kind == "objective":
        c = _scan(kind, "", nx, ny, nz, vx, cols, rows, du, views, lam=1e-3, dtype=rng.choice(["f32", "f16", "bf16"]))
    else:
        # no axial truncation: the detector covers the volume from every view
        near = DSO - 0.5 * vx * math.hypot(nx, ny)
        rows = int((DSO - DOD) / near * vx * nz / du) + rng.randint(4, 12)
        c = _scan(kind, "", nx, ny, nz, vx, cols, rows, du, _log_int(rng, 30, 240),
                  window=rng.choice(["ramp", "hann"]), dtype=rng.choice(["f32", "f32", "f16", "bf16"]))
    del c["name"]
    return c


# -------------------------------------------------------------------- inputs
def _geometry(c):
    return Geometry(nx=c["nx"], ny=c["ny"], nz=c["nz"], vx=c["vx"], ncols=c["cols"], nrows=c["rows"], du=c["du"],
                    dv=c["dv"], nviews=c["views"], dso=DSO, dod=DOD, nsources=c["sources"], src_z0=c["src_z0"],
                    src_dz=c["src_dz"], style=c["style"])


def _scene(c, seed):
    # the ten ellipsoids, scaled to the volume's width
    return ellipsoid_params(seed, 10, 0.9 * c["vx"] * min(c["nx"], c["ny"]) / 128.0)


def _centres(c, dtype):
    def axis(n):
        return (torch.arange(n, device=DEVICE, dtype=dtype) + (0.5 - n / 2.0)) * c["vx"]
    return axis(c["nx"])[None, None, :], axis(c["ny"])[None, :, None], axis(c["nz"])[:, None, None]


def _phantom(c, seed, noise):
    """The scene on the voxel grid, FP32, with Gaussian noise of `noise` /mm."""
    x, y, z = _centres(c, torch.float32)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    out = torch.randn((c["nz"], c["ny"], c["nx"]), device=DEVICE, generator=gen).mul_(noise)
    centre, axes, angle, mu = _scene(c, seed)
    for e in range(10):
        rt = rotation_zyz(*angle[e]).T / axes[e][:, None]
        px, py, pz = x - float(centre[e][0]), y - float(centre[e][1]), z - float(centre[e][2])
        q = 0.0
        for r in range(3):
            q = q + (float(rt[r, 0]) * px + float(rt[r, 1]) * py + float(rt[r, 2]) * pz) ** 2
        out += (q <= 1.0).to(torch.float32) * float(mu[e])
    return out


def _view_rays(c, v, dtype=torch.float32):
    """Pixel positions and source positions of view v: (x1, y1, z1), (x2, y2, z2)
    broadcastable to [source, row, column]."""
    s, cs = _angle(c, v)
    u = (torch.arange(c["cols"], device=DEVICE, dtype=dtype) + (0.5 - c["cols"] / 2.0)) * c["du"]
    w = (torch.arange(c["rows"], device=DEVICE, dtype=dtype) + (0.5 - c["rows"] / 2.0)) * c["dv"]
    u, w = u[None, None, :], w[None, :, None]
    x1, y1, z1 = DOD * cs - u * s, DOD * s + u * cs, w
    if c["style"] == 2:
        x2, y2 = DSO * cs - u * s, DSO * s + u * cs
    else:
        x2, y2 = torch.full_like(u, DSO * cs), torch.full_like(u, DSO * s)
    if c["style"] == 0:
        z2 = c["src_z0"] + c["src_dz"] * torch.arange(c["sources"], device=DEVICE, dtype=dtype)[:, None, None]
    else:
        z2 = w
    return (x1, y1, z1), (x2, y2, z2)


def _angle(c, v, sign=-1.0):
    """(sin, cos) of view v: single-precision angles and tables, as the
    projectors document them."""
    f = np.float32
    th = f(f(f(v) * f(360.0 / c["views"])) * f(math.pi) / f(180.0)) * f(sign)
    return float(f(math.sin(float(th)))), float(f(math.cos(float(th))))


def _measurements(c, seed):
    """Noisy line integrals of the scene, FP32 [view, (source,) row, column]."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    centre, axes, angle, mu = _scene(c, seed)
    out = torch.empty((c["views"], c["sources"], c["rows"], c["cols"]), device=DEVICE)
    for v in range(c["views"]):
        p1, p2 = _view_rays(c, v)
        d = [b - a for a, b in zip(p1, p2)]
        dist = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
        acc = out[v]
        acc.zero_()
        for e in range(10):
            rt = rotation_zyz(*angle[e]).T / axes[e][:, None]
            o = [a - float(k) for a, k in zip(p1, centre[e])]
            w = [float(rt[r, 0]) * o[0] + float(rt[r, 1]) * o[1] + float(rt[r, 2]) * o[2] for r in range(3)]
            t = [float(rt[r, 0]) * d[0] + float(rt[r, 1]) * d[1] + float(rt[r, 2]) * d[2] for r in range(3)]
            a = t[0] * t[0] + t[1] * t[1] + t[2] * t[2]
            b = (w[0] * t[0] + w[1] * t[1] + w[2] * t[2]) / a
            n = [w[r] - b * t[r] for r in range(3)]
            disc = 1.0 - (n[0] * n[0] + n[1] * n[1] + n[2] * n[2])
            acc += 2.0 * float(mu[e]) * dist * torch.sqrt(disc.clamp_(min=0.0) / a)
        counts = torch.poisson(I0 * torch.exp(-acc), generator=gen)
        torch.log_(counts.clamp_(min=1.0).div_(I0))
        acc.copy_(counts.neg_())
    return out if c["sources"] > 1 else out[:, 0].contiguous()


def _inputs(c, seed):
    dt = DTYPES[c["dtype"]]
    if c["kind"] == "tv_fgp":
        return SimpleNamespace(x=_phantom(c, seed, 0.002).to(dt))
    if c["kind"] == "fdk":
        return SimpleNamespace(meas=_measurements(c, seed).to(dt))
    n = SimpleNamespace(x=_phantom(c, seed, 0.0005).to(dt), meas=_measurements(c, seed))
    if c["kind"] == "iteration":
        n.x_prev = _phantom(c, seed, 0.001).to(dt)
        n.meas = n.meas.to(dt)
    return n


def prepare(case, seed):
    st = _inputs(case, seed)
    st.case, st.ct = case, Context(0)
    if case["kind"] != "tv_fgp":
        st.g = _geometry(case)
    if case["kind"] in ("sart", "iteration", "tv_fgp"):
        st.out = torch.empty_like(st.x)
        st.out_prev = torch.empty_like(st.x) if case["kind"] == "iteration" else None
    if case["kind"] == "gradient":
        st.x.requires_grad_(True)
        if "lam" in case:
            st.lam = torch.tensor(case["lam"], device=DEVICE, dtype=torch.float64)
    return st


# ---------------------------------------------------------------------- pass
def run(state):
    c, ct, kind = state.case, state.ct, state.case["kind"]
    if kind == "sart":
        state.out.copy_(state.x)
        return ct.sart_sweep(state.g, state.out, state.meas, beta=c["beta"], subset=c["subset"], order=c["order"])
    if kind == "iteration":
        state.out.copy_(state.x)
        state.out_prev.copy_(state.x_prev)
        t = ct.sart_fista_iteration(state.g, state.out, state.out_prev, state.meas, 2.5, beta=c["beta"],
                                    subset=c["subset"], order=c["order"], fgp_lambda=c["lam"], fgp_niter=c["inner"])
        return state.out, state.out_prev, t
    if kind == "gradient":
        p = project(state.x, state.g, ct, out_dtype=torch.float32)
        residual = p.detach() - state.meas
        if "lam" not in c:
            return p.detach(), torch.autograd.grad(p, state.x, residual)[0]
        tv = tv_eps(state.x, EPS, ct)
        return p.detach(), tv.detach(), torch.autograd.grad((p, tv), state.x, (residual, state.lam))[0]
    if kind == "objective":
        return ct.objective(state.g, state.x, state.meas, c["lam"])
    if kind == "tv_fgp":
        state.out.copy_(state.x)
        return ct.tv_fgp(state.out, c["lam"], c["inner"])
    return ct.fdk(state.g, state.meas, window=c["window"])


def work(case):
    c = case
    vox = c["nx"] * c["ny"] * c["nz"]
    es = 4 if c["dtype"] == "f32" else 2
    if c["kind"] == "tv_fgp":
        # the volume in and out; ~45 operations per voxel and inner iteration
        return {"bytes": 2 * vox * es, "flops": 45 * vox * c["inner"]}
    rays = c["views"] * c["sources"] * c["rows"] * c["cols"]
    # a segment per crossed voxel (multiply-add) for each ray through the
    # volume; a chord per (voxel, footprint pixel)
    seg = 2 * rays * int(1.3 * max(c["nx"], c["ny"]))
    mag = 1.0 if c["style"] == 2 else (DSO - DOD) / DSO
    foot = (1.27 * mag * c["vx"] / c["du"] + 1) * ((mag if c["style"] == 0 else 0.0) * c["vx"] / c["dv"] + 1)
    images = c["views"] * c["sources"]
    chord = 5 * vox * 0.785 * foot * images
    if c["kind"] == "fdk":
        pad = 2 * c["cols"]
        return {"bytes": rays * es + vox * es, "flops": 10 * vox * c["views"] + rays * 5 * math.log2(pad) * 2}
    if c["kind"] == "sart":
        return {"bytes": 4 * rays + 2 * vox * es, "flops": seg + chord}
    if c["kind"] == "iteration":
        return {"bytes": es * rays + 4 * vox * es, "flops": seg + chord + 45 * vox * c["inner"]}
    if c["kind"] == "gradient":
        seen = min(1.0, c["rows"] * c["dv"] / (1.5 * c["nz"] * c["vx"]))
        return {"bytes": 8 * rays + 2 * vox * es, "flops": seg + 2 * vox * seen * foot * images}
    return {"bytes": 4 * rays + vox * es, "flops": seg}


# ----------------------------------------------------------- 64-bit reference
def _segments(c, p1, p2, visit):
    """Calls visit(rays, voxel, length) for the segments of flat rays p1 -> p2:
    the rays are walked slab by slab along their main lateral axis, in which a
    slab holds at most one crossing of each other axis.  Returns the rays'
    lengths inside the volume."""
    n = (c["nx"], c["ny"], c["nz"])
    v = c["vx"]
    b = [-v * k / 2.0 for k in n]
    e = [q - a for a, q in zip(p1, p2)]
    lo = torch.zeros_like(p1[0])
    hi = torch.ones_like(lo)
    for k in range(3):
        a0, a1 = (b[k] - p1[k]) / e[k], (b[k] + v * n[k] - p1[k]) / e[k]
        par = e[k].abs() < 1e-6 * v
        inside = (p1[k] >= b[k]) & (p1[k] <= b[k] + v * n[k])
        a0 = torch.where(par, torch.where(inside, -math.inf, math.inf), a0)
        a1 = torch.where(par, torch.where(inside, math.inf, -math.inf), a1)
        lo, hi = torch.maximum(lo, torch.minimum(a0, a1)), torch.minimum(hi, torch.maximum(a0, a1))
    hi = torch.maximum(hi, lo)
    dist = torch.sqrt(e[0] ** 2 + e[1] ** 2 + e[2] ** 2)
    main_x = e[0].abs() >= e[1].abs()
    for m, o, sel in ((0, 1, main_x), (1, 0, ~main_x)):
        r = torch.nonzero(sel & (hi > lo)).flatten()
        if r.numel() == 0:
            continue
        q = [p1[k][r] for k in range(3)]
        d = [e[k][r] for k in range(3)]
        rl, rh, rd = lo[r], hi[r], dist[r]
        for i in range(n[m]):
            a0, a1 = (b[m] + i * v - q[m]) / d[m], (b[m] + (i + 1) * v - q[m]) / d[m]
            s = torch.maximum(torch.minimum(a0, a1), rl)
            t = torch.maximum(torch.minimum(torch.maximum(a0, a1), rh), s)
            cuts = []
            for k in (o, 2):
                f0 = torch.floor((q[k] + s * d[k] - b[k]) / v)
                f1 = torch.floor((q[k] + t * d[k] - b[k]) / v)
                cut = (b[k] + torch.maximum(f0, f1) * v - q[k]) / d[k]
                cuts.append(torch.where(f0 == f1, t, torch.minimum(torch.maximum(cut, s), t)))
            stops = [s, torch.minimum(*cuts), torch.maximum(*cuts), t]
            for s0, s1 in zip(stops, stops[1:]):
                mid = 0.5 * (s0 + s1)
                j = torch.floor((q[o] + mid * d[o] - b[o]) / v).clamp_(0, n[o] - 1).long()
                k = torch.floor((q[2] + mid * d[2] - b[2]) / v).clamp_(0, n[2] - 1).long()
                x, y = (i, j) if m == 0 else (j, i)
                visit(r, (k * n[1] + y) * n[0] + x, (s1 - s0) * rd)
    return (hi - lo) * dist


def _chunks(c, views):
    """(views, flat rays) in portions of about four million rays."""
    per = max(1, 4000000 // (c["sources"] * c["rows"] * c["cols"]))
    shape = (c["sources"], c["rows"], c["cols"])
    for k in range(0, len(views), per):
        part = views[k:k + per]
        rays = [_view_rays(c, v, torch.float64) for v in part]
        yield part, [[torch.cat([r[s][a].expand(shape).reshape(-1) for r in rays]) for a in range(3)]
                     for s in range(2)]


def _ray_sums(c, x, views):
    """Ray sums and ray lengths of the views, [view, source, row, column]."""
    flat = x.flatten()
    sums, lens = [], []
    for part, (p1, p2) in _chunks(c, views):
        acc = torch.zeros_like(p1[0])

        def visit(r, vox, seg, acc=acc):
            acc[r] += seg * flat[vox]
        ln = _segments(c, p1, p2, visit)
        shape = (len(part), c["sources"], c["rows"], c["cols"])
        sums.append(torch.where(ln < 1e-6 * c["vx"], 0.0, acc).view(shape))
        lens.append(ln.view(shape))
    return torch.cat(sums), torch.cat(lens)


def _transpose(c, y, views):
    out = torch.zeros(c["nx"] * c["ny"] * c["nz"], device=DEVICE, dtype=torch.float64)
    k = 0
    for part, (p1, p2) in _chunks(c, views):
        w = y[k:k + len(part)].reshape(-1)
        k += len(part)
        _segments(c, p1, p2, lambda r, vox, seg, w=w: out.index_add_(0, vox, seg * w[r]))
    return out.view(c["nz"], c["ny"], c["nx"])


def _chord_sums(c, v, corr, W, L):
    """Adds view v's sums of chord x correction and of chords to W and L."""
    s, cs = _angle(c, v)
    h, dv, du, rows, cols, style = c["vx"] / 2.0, c["dv"], c["du"], c["rows"], c["cols"], c["style"]
    umin, wmin = (0.5 - cols / 2.0) * du, (0.5 - rows / 2.0) * dv
    X, Y, Z = _centres(c, torch.float64)
    us, rs = [], []
    for a in (-h, h):
        for b in (-h, h):
            t = (X + a) * cs + (Y + b) * s
            q = -(X + a) * s + (Y + b) * cs
            rs.append((t - DOD) / (DSO - t))
            us.append(q if style == 2 else (rs[-1] + 1.0) * q)
    us, rs = torch.stack(us), torch.stack(rs)
    y0 = torch.floor((us.amin(0) - umin) / du + 0.5)
    y1 = torch.floor((us.amax(0) - umin) / du + 0.5)
    spans = []
    for cc in range(int((y1 - y0).max()) + 1):
        col = y0 + cc
        u = umin + col * du
        qx, qy = DOD * cs - u * s, DOD * s + u * cs
        ex = (DSO * cs - u * s if style == 2 else DSO * cs) - qx
        ey = (DSO * s + u * cs if style == 2 else DSO * s) - qy
        ax, bx = (X - h - qx) / ex, (X + h - qx) / ex
        ay, by = (Y - h - qy) / ey, (Y + h - qy) / ey
        lo = torch.maximum(torch.minimum(ax, bx), torch.minimum(ay, by))
        hi = torch.minimum(torch.maximum(ax, bx), torch.maximum(ay, by))
        ok = (col <= y1) & (col >= 0) & (col < cols)
        spans.append((lo, torch.where(ok, hi, -math.inf), ex * ex + ey * ey, col.clamp(0, cols - 1).long()))
    flat = corr.reshape(-1)
    step = max(1, 40000000 // (c["nx"] * c["ny"]))
    for k in range(0, c["nz"], step):
        z = Z[k:k + step]
        if style == 0:
            w = [r * (z + f - c["src_z0"]) + z + f for f in (-h, h) for r in (rs.amin(0), rs.amax(0))]
            z0 = torch.floor((torch.minimum(w[0], w[1]) - wmin) / dv + 0.5)
            z1 = torch.floor((torch.maximum(w[2], w[3]) - wmin) / dv + 0.5)
        else:
            z0 = torch.floor((z - wmin) / dv + 0.5)
            z1 = z0
        for rr in range(int((z1 - z0).max()) + 1):
            row = z0 + rr
            ez = (c["src_z0"] if style == 0 else z) - (wmin + row * dv)
            az, bz = (z - h - (wmin + row * dv)) / ez, (z + h - (wmin + row * dv)) / ez
            zl, zh = torch.minimum(az, bz), torch.maximum(az, bz)
            on = (row <= z1) & (row >= 0) & (row < rows)
            base = row.clamp(0, rows - 1).long() * cols
            for lo, hi, e2, col in spans:
                ln = torch.sqrt(e2 + ez * ez) * (torch.minimum(hi, zh) - torch.maximum(lo, zl))
                ln = torch.where(on & (ln > 1e-6 * c["vx"]), ln, 0.0)
                W[k:k + step] += ln * flat[base + col]
                L[k:k + step] += ln


def _exact_sart(c, n):
    x, meas = n.x.double(), n.meas.double()
    views, size = c["views"], c["subset"]
    nsub = (views + size - 1) // size
    if c["order"] == "interleaved" and size > 1:
        subsets = [list(range(s, views, nsub)) for s in range(nsub)]
    else:
        subsets = [list(range(k, min(k + size, views))) for k in range(0, views, size)]
    X, Y, _ = _centres(c, torch.float64)
    mask = X * X + Y * Y >= (c["nx"] - 1) * (c["ny"] - 1) * c["vx"] ** 2 / 4.0
    for sub in subsets:
        sums, ln = _ray_sums(c, x, sub)
        corr = torch.where(ln[:, 0] < 1e-6 * c["vx"], 0.0, (meas[sub] - sums[:, 0]) / ln[:, 0])
        W, L = torch.zeros_like(x), torch.zeros_like(x)
        for k, v in enumerate(sub):
            _chord_sums(c, v, corr[k], W, L)
        x = torch.where((L < 1e-6 * c["vx"]) | mask, x, x + c["beta"] * W / L)
    return x


def _exact_fgp(x, lam, inner):
    def shift(p, axis):   # p of the lower neighbour, zero outside
        out = torch.zeros_like(p)
        out.narrow(axis, 1, p.shape[axis] - 1).copy_(p.narrow(axis, 0, p.shape[axis] - 1))
        return out

    def residual(duals):
        return x - lam * sum(p - shift(p, ax) for p, ax in zip(duals, (2, 1, 0)))
    r = [torch.zeros_like(x) for _ in range(3)]
    old = [torch.zeros_like(x) for _ in range(3)]
    t = 1.0
    for _ in range(inner):
        d = residual(r)
        for p, ax in zip(r, (2, 1, 0)):
            m = x.shape[ax] - 1
            p.narrow(ax, 0, m).add_(d.narrow(ax, 0, m) - d.narrow(ax, 1, m), alpha=1.0 / (12.0 * lam))
        norm = torch.sqrt(r[0] ** 2 + r[1] ** 2 + r[2] ** 2).clamp_(min=1.0)
        t1 = (1.0 + math.sqrt(1.0 + 4.0 * t * t)) / 2.0
        new = [p / norm for p in r]
        r = [a + (t - 1.0) / t1 * (a - b) for a, b in zip(new, old)]
        old, t = new, t1
    return residual(old)


def _exact_fdk(c, meas):
    pad = 2 * c["cols"]
    k = torch.fft.fftfreq(pad, 1.0 / pad, device=DEVICE, dtype=torch.float64)
    H = 0.5 * k.abs() / (2.0 * c["du"] * DSO / (DSO - DOD)) / (pad // 2)
    if c["window"] == "hann":
        H = H * 0.5 * (1.0 + torch.cos(2.0 * math.pi * k / pad))
    u = (torch.arange(c["cols"], device=DEVICE, dtype=torch.float64) + (0.5 - c["cols"] / 2.0)) * c["du"]
    w = (torch.arange(c["rows"], device=DEVICE, dtype=torch.float64) + (0.5 - c["rows"] / 2.0)) * c["dv"]
    iso = DSO / (DSO - DOD)
    cosw = DSO / torch.sqrt(DSO ** 2 + (u * iso)[None, :] ** 2 + (w * iso)[:, None] ** 2)
    X, Y, Z = _centres(c, torch.float64)
    X, Y = X[0], Y[0]
    out = torch.zeros((c["nz"], c["ny"], c["nx"]), device=DEVICE, dtype=torch.float64)
    for v in range(c["views"]):
        img = torch.fft.ifft(torch.fft.fft(meas[v].double() * cosw, n=pad) * H).real[:, :c["cols"]].reshape(-1)
        s, cs = _angle(c, v, 1.0)
        inv = 1.0 / (DSO + X * s - Y * cs)
        p = ((X * cs + Y * s) * (DSO - DOD) * inv - float(u[0])) / c["du"]
        ksi = (Z * ((DSO - DOD) * inv) - float(w[0])) / c["dv"]
        ok = (ksi >= 0) & (ksi + 1 < c["rows"]) & ((p >= 0) & (p + 1 < c["cols"]))
        kf, pf = torch.floor(ksi), torch.floor(p)
        i = kf.clamp(0, c["rows"] - 2).long() * c["cols"] + pf.clamp(0, c["cols"] - 2).long()
        a, b = ksi - kf, p - pf
        val = (1.0 - a) * ((1.0 - b) * img[i] + b * img[i + 1]) + \
            a * ((1.0 - b) * img[i + c["cols"]] + b * img[i + c["cols"] + 1])
        out += torch.where(ok, (DSO * inv) ** 2 * (2.0 * math.pi / c["views"]) * val, 0.0)
    return out


def _tv(x):
    q = torch.zeros_like(x)
    for ax in range(3):
        m = x.shape[ax] - 1
        q.narrow(ax, 0, m).add_((x.narrow(ax, 0, m) - x.narrow(ax, 1, m)) ** 2)
    return float(torch.sqrt(q).sum())


def exact(case, seed):
    c, kind = case, case["kind"]
    vox = c["nx"] * c["ny"] * c["nz"]
    if kind == "iteration":
        return None   # a chain of stochastically rounded updates
    if kind == "tv_fgp":
        return _exact_fgp(_inputs(c, seed).x.double(), c["lam"], c["inner"])
    steps = c["views"] * c["sources"] * c["rows"] * c["cols"] * max(c["nx"], c["ny"])
    if kind == "fdk":
        return _exact_fdk(c, _inputs(c, seed).meas) if vox * c["views"] < 6e10 else None
    if kind == "sart":
        if c["dtype"] != "f32" or steps > 1.5e10 or vox * c["views"] > 2.5e9:
            return None
        return _exact_sart(c, _inputs(c, seed))
    if steps > 3e10:
        return None
    n = _inputs(c, seed)
    x, views = n.x.double(), list(range(c["views"]))
    sums, _ = _ray_sums(c, x, views)
    diff = sums - n.meas.double().view_as(sums)
    if kind == "objective":
        data, tv = float((diff * diff).sum()), _tv(x)
        return data, tv, data + 2.0 * c["lam"] * tv
    grad = _transpose(c, diff, views)
    if "lam" not in c:
        return sums.view(n.meas.shape), grad
    x.requires_grad_(True)
    q = torch.full_like(x, EPS)
    for ax in range(3):
        q = q + torch.nn.functional.pad(x.diff(dim=ax), [0, 0] * (2 - ax) + [1, 0]) ** 2
    tv = torch.sqrt(q).sum()
    tv.backward()
    return sums.view(n.meas.shape), tv.detach(), grad + c["lam"] * x.grad
