"""Scratch that only makes a call faster (copies of the volume, partial sums) is
not needed for its result: the calls run where that scratch cannot be had, be
it that the memory is not there or that the stream is being captured into a
graph.  Against the CPU oracle at the parity bars (1e-5 on projections, 1e-4 on
reconstructions)."""
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


def rel(a, b):
    b = np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a.double().cpu().numpy() - b) / max(np.linalg.norm(b), 1e-300))


def captured(fn):
    """fn captured into a graph after what warmed its context up; replays it."""
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


@pytest.fixture
def fresh():
    torch.cuda.empty_cache()
    c = Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


def test_ray_sums_without_transposed_copy(fresh):
    """A context that has walked views along x only captures views along y."""
    g = Geometry(nx=96, ny=92, nz=80, vx=1.0, ncols=512, nrows=530, du=0.33, dv=150.0 / 530, nviews=12,
                 angle_step_deg=10.0)
    x = phantom(g, seed=2, scale=0.3)
    xd = x.cuda()
    fresh.forward(g, xd, view0=0, nviews=4)
    out = torch.zeros((4, g.nrows, g.ncols), device="cuda")
    graph = captured(lambda: fresh.forward(g, xd, out, view0=8, nviews=4))
    ref = orc.forward(g, x.numpy(), prec=32)[8:]
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel(out, ref) <= 1e-5
    fresh.forward(g, xd, out, view0=8, nviews=4)   # with the copy
    assert rel(out, ref) <= 1e-5


def test_planar_sweep_without_copy(fresh):
    """A context that has run the BF16 fan sweep, which needs no copy, captures
    the FP32 one."""
    g = Geometry(nx=25, ny=27, nz=21, vx=1.0, ncols=41, nrows=21, du=1.1, dv=1.0, nviews=9, dso=90.0, dod=-45.0,
                 angle_step_deg=37.3, style=1)
    x = phantom(g, seed=2, scale=0.3).numpy()
    b = orc.forward(g, x, prec=32)
    x0 = (0.7 * x + 0.004).astype(np.float32)
    ref = orc.sart_sweep(g, x0, b, beta=0.8, subset=1, order="ascending", prec=32)
    start, bd = torch.as_tensor(x0).cuda(), torch.as_tensor(b).float().cuda()
    fresh.sart_sweep(g, start.bfloat16(), bd, beta=0.8, subset=1)
    v = start.clone()
    graph = captured(lambda: fresh.sart_sweep(g, v, bd, beta=0.8, subset=1))
    for _ in range(3):
        v.copy_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert rel(v, ref) <= 1e-4
    v.copy_(start)
    fresh.sart_sweep(g, v, bd, beta=0.8, subset=1)   # with the copy
    assert rel(v, ref) <= 1e-4


def test_adjoint_without_parts(fresh):
    """A context whose tables hold the views but not the parts' sums captures
    the gather of many views on few tiles; 2e-5 as a 1 mm voxel spans 7.4e-3 of
    a ray's alpha, whose two crossings round to 6e-8 each."""
    g = Geometry(nx=25, ny=21, nz=9, vx=1.0, ncols=41, nrows=29, du=1.1, nviews=20, dso=90.0, dod=-45.0,
                 angle_step_deg=37.3)
    wide = replace(g, ncols=80, nrows=60)   # 7 views, in one part: larger tables than 20 views of g
    y = np.random.default_rng(3).standard_normal(g.proj_shape)
    yd = torch.as_tensor(y).float().cuda()
    fresh.adjoint(wide, torch.zeros((7, 60, 80), device="cuda"), view0=0, nviews=7)
    out = torch.zeros(g.vol_shape, device="cuda")
    graph = captured(lambda: fresh.adjoint(g, yd, out))
    ref = orc.adjoint(g, y, prec=32)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert rel(out, ref) <= 2e-5
    fresh.adjoint(g, yd, out)   # in parts
    assert rel(out, ref) <= 2e-5


def test_objective_without_copies(fresh):
    """The objective of a 1.9 GiB volume with room for both copies of it, for
    one and for none: the same sums to 4e-5 (1e-5 on Ax, which enters squared,
    each way)."""
    g = Geometry(nx=640, ny=640, nz=1200, vx=0.4, ncols=256, nrows=256, du=1.2, dv=0.4, nviews=8)
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand(g.vol_shape, device="cuda", generator=gen).mul_(0.02)
    meas = torch.rand(g.proj_shape, device="cuda", generator=gen)
    nbytes = g.nvox * 4
    scratch = core.lib().ct_scratch_bytes
    scratch.argtypes, scratch.restype = [ctypes.c_void_p], ctypes.c_size_t
    values = []
    for copies, spare in ((2, None), (1, nbytes + (1 << 30)), (0, 1 << 30)):
        c = Context(0)
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        fill = None
        if spare is not None:
            fill = torch.empty(torch.cuda.mem_get_info()[0] - spare, device="cuda", dtype=torch.uint8)
        try:
            values.append(c.objective(g, x, meas, 1e-3))
            assert scratch(c._h) // nbytes == copies
        finally:
            c.close()
            del fill
            torch.cuda.empty_cache()
    for v in values[1:]:
        assert all(abs(p - q) <= 4e-5 * abs(q) for p, q in zip(v, values[0])), values
