"""The column walk (one workgroup per detector column) of launches large enough
to take it, from 3 * 2^24 (ray, x/y plane) pairs on, twice that for the
objective: small geometries with as many views as that needs, in all three
storage types.  Ray sums and corrections assert that they took the walk by the
copies of the volume in their context's scratch.

Bars against the FP32 oracle on the stored volume: 1e-5 on ray sums, 2e-5 on
corrections (as much again from the chord lengths), 4e-5 on the objective (the
1e-5 of Ax enters squared, and b = Ax/2 + 0.01)."""
import ctypes
from dataclasses import replace

import numpy as np
import pytest
import torch

from gpu_amd import core
from gpu_amd.core import Context
from gpu_amd.geometry import Geometry
from gpu_amd.phantom import phantom
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

PAIRS = 3 << 24
DTYPES = [torch.float32, torch.float16, torch.bfloat16]
SMALL = Geometry(nx=24, ny=20, nz=16, vx=1.0, ncols=40, nrows=28, du=1.1, nviews=9, dso=90.0, dod=-45.0,
                 angle_step_deg=37.3)


def rel(a, b):
    a, b = a.double().cpu().numpy(), np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def with_pairs(g, pairs):
    per = g.ncols * g.nrows * g.nsources * (g.nx + g.ny)
    return replace(g, nviews=-(-pairs // per))


def copies(c, g, dt):
    """z-quad copies of the volume that context c holds."""
    fn = core.lib().ct_scratch_bytes
    fn.argtypes, fn.restype = [ctypes.c_void_p], ctypes.c_size_t
    return (fn(c._h) - 8 * g.nviews) // (g.nx * g.ny * (g.nz + 3 & ~3) * torch.finfo(dt).bits // 8)


def check(g, dt, seed):
    x = phantom(g, seed=seed, scale=0.3, device="cuda").to(dt)
    xs = x.float().cpu().numpy()

    def on_fresh(call):
        c = Context(0)
        try:
            out = call(c)
            torch.cuda.synchronize()
            return out, copies(c, g, dt)
        finally:
            c.close()

    g = with_pairs(g, PAIRS)
    ref = orc.forward(g, xs, prec=32)
    got, n = on_fresh(lambda c: c.forward(g, x, out_dtype=torch.float32))
    assert n == 2 and rel(got, ref) <= 1e-5

    # b = 2 Ax + 0.01 keeps b - 0.9 Ax away from cancellation
    y = (x.float() * 0.9).to(dt)
    meas = (2.0 * ref + 0.01).astype(np.float32)
    want = orc.sart_correction(g, y.float().cpu().numpy(), meas, view0=0, nviews=g.nviews, prec=32)
    md = torch.as_tensor(meas).cuda()
    got, n = on_fresh(lambda c: c.sart_correction(g, y, md, view0=0, nviews=g.nviews))
    # as residuals, times the oracle's chord lengths, of rays with chords of 0.01
    # mm and more: a crossing rounds to 1.2e-7 of the ray's 135 mm, so that
    # among a million rays a few with shorter chords would be all of the norm
    chord = orc.forward(g, np.ones_like(xs), prec=32).reshape(want.shape)
    chord[chord < 0.01] = 0.0
    # (BF16 corrections walk views along y by ray, without the transposed copy)
    assert n == (1 if dt == torch.bfloat16 else 2)
    assert rel(got.view(want.shape) * torch.as_tensor(chord).cuda(), want * chord) <= 2e-5

    g = with_pairs(g, 2 * PAIRS)
    ref = orc.forward(g, xs, prec=32)
    meas = (0.5 * ref + 0.01).astype(np.float32)
    md = torch.as_tensor(meas).cuda()
    (data, _, _), _ = on_fresh(lambda c: c.objective(g, x, md))
    want = float(((ref.astype(np.float64) - meas) ** 2).sum())
    assert abs(data - want) <= 4e-5 * want


@pytest.mark.parametrize("nrows", [1, 64, 65, 128, 129, 256, 257])
@pytest.mark.parametrize("dt", DTYPES)
def test_row_blocks(dt, nrows):
    """Rows of a column in blocks of 128 or 256 and part blocks; an odd detector
    on an even volume has rays in the planes between voxels."""
    check(replace(SMALL, nrows=nrows, dv=30.8 / nrows, ncols=21), dt, 5)


@pytest.mark.parametrize("kw", [
    dict(x_offset=3, det_offset=2.2, ncols=37, nrows=21),
    dict(nx=17, ny=23, nz=11, vx=0.9, vy=1.2, vz=0.7, du=0.8, dv=1.3),
    dict(nsources=4, src_z0=-9.0, src_dz=6.0, nrows=12),
    dict(style=1, nrows=16, dv=1.0),
    dict(style=2, nrows=16, dv=1.0, det_offset=0.7, x_offset=1),
], ids=["offsets", "aniso", "multisource", "fan", "parallel"])
@pytest.mark.parametrize("dt", DTYPES)
def test_geometries(dt, kw):
    check(replace(SMALL, **kw), dt, 11)


@pytest.mark.parametrize("kw", [
    dict(nz=6, vz=0.7, ncols=11, nrows=17, dv=1.1146163743152828, nsources=5, src_z0=-12.0, src_dz=6.0),
    dict(nz=58, vz=0.35, ncols=21, nrows=41, dv=0.30271779082383904),
], ids=["five sources", "one source"])
@pytest.mark.parametrize("dt", DTYPES)
def test_level_rays(dt, kw):
    """A middle row that lies level with a source, to rounding in the plane
    between two slices: the whole row belongs to the slab that the reference's
    set-up puts it in."""
    check(replace(SMALL, **kw), dt, 5)
