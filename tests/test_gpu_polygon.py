"""Caller-supplied polygons (z2d_gpu_fill_polygon, z2d_gpu_batch_fill_polygon):
edges taken as they are, also those that no sample row meets (horizontal ones
on and between sample rows and at the borders of bands, and ones with a NaN
end), in few and many edge groups and over more than eight bands, after draws
that left other edges in the same buffers; equal to the oracle's rasterizer,
whose active-edge test passes such edges by."""
import ctypes as C

import numpy as np
import pytest

from z2d_amd import abi, scenes
from gpu_util import diff_report, gpu_backend
from oracle_backend import lib as oracle_lib
from zscene import Surface

pytestmark = pytest.mark.gpu

W, H = 90, 200  # 13 bands of 16 rows


def _polygon(rng, n, scale):
    """The edges of a closed polygon of n points in the scaled space
    (Polygon.addEdge) and their extents (top, bottom, left, right)."""
    p = np.array([(rng.uniform(-4, W + 4), rng.uniform(-4, H + 4)) for _ in range(n)]) * scale
    q = np.roll(p, -1, axis=0)
    e = np.zeros(n, abi.EDGE_DTYPE)
    e["y0"], e["y1"] = p[:, 1], q[:, 1]
    e["x_start"] = np.where(p[:, 1] < q[:, 1], p[:, 0], q[:, 0])
    e["x_inc"] = (q[:, 0] - p[:, 0]) / (q[:, 1] - p[:, 1])
    return e, (p[:, 1].min(), p[:, 1].max(), p[:, 0].min(), p[:, 0].max())


def _with_idle(rng, edges, kind, scale):
    """The polygon with edges between its own that no sample row meets."""
    idle = np.zeros(max(3, len(edges) // 2), abi.EDGE_DTYPE)
    y = np.array([rng.randint(0, H) * scale for _ in idle], float)
    if kind == "horizontal":
        # between sample rows, on one, on a band's border
        y[1::3] += 0.5
        y[2::3] = y[2::3] // (16 * scale) * (16 * scale)
        idle["y0"] = idle["y1"] = y
    else:
        idle["y0"], idle["y1"] = y, y[::-1]
        idle["y0" if kind == "nan_y0" else "y1"] = np.nan
    idle["x_start"] = [rng.uniform(0, W * scale) for _ in idle]
    idle["x_inc"] = [rng.uniform(-2, 2) for _ in idle]
    at = np.sort([rng.randint(0, len(edges)) for _ in idle])
    return np.insert(edges, at, idle)


def _leave_edges(fill):
    """A draw of many edges in all bands."""
    nodes = scenes.star_512()["draws"][0][1].copy()
    nodes["v"][:, 0] *= W / 512
    nodes["v"][:, 1] *= H / 512
    nodes = np.concatenate([nodes[:-1]] * 60 + [nodes[-1:]])
    assert fill(abi.solid_pattern(abi.rgba(9, 8, 7, 255)), nodes, abi.fill_opts()) == 0


@pytest.mark.parametrize("kind", ["none", "horizontal", "nan_y0", "nan_y1"])
@pytest.mark.parametrize("n", [3, 40, 64, 65, 190])
@pytest.mark.parametrize("aa,op", [(abi.AA_DEFAULT, "src_over"), (abi.AA_NONE, "src_over"),
                                   (abi.AA_SUPERSAMPLE_4X, "src_over"), (abi.AA_DEFAULT, "src_in"),
                                   (abi.AA_NONE, "src_in")],
                         ids=["msaa", "none", "ssaa", "msaa-unbounded", "none-unbounded"])
def test_polygon(kind, n, aa, op):
    from z2d_amd import gpu
    be = gpu_backend()
    L = gpu.lib()
    rng = scenes.SplitMix64(0x9017 + n)
    scale = 1.0 if aa == abi.AA_NONE else 4.0
    edges, ext = _polygon(rng, n, scale)
    if kind != "none":
        edges = _with_idle(rng, edges, kind, scale)
    ext = (C.c_double * 4)(*ext)
    pat = abi.solid_pattern(abi.rgba(60, 20, 90, 110))
    init = np.full(W * H * 4, 255, np.uint8)
    for rule in (abi.NON_ZERO, abi.EVEN_ODD):
        args = (aa, rule, abi.OP[op], abi.PRECISION_INTEGER)
        want = Surface(abi.RGBA, W, H)
        want.buf[:want.nbytes] = init
        d = want.desc()
        assert oracle_lib().zo_fill_polygon(C.byref(d), C.byref(pat), edges.ctypes.data,
                                            len(edges), ext, *args) == 0
        # one painter call after another's
        got, other = Surface(abi.RGBA, W, H), Surface(abi.RGBA, W, H)
        got.buf[:got.nbytes] = init
        _leave_edges(lambda *a: be.fill(other, *a))
        d = got.desc()
        assert L.z2d_gpu_fill_polygon(be.ctx.h, C.byref(d), C.byref(pat), edges.ctypes.data,
                                      len(edges), ext, *args) == 0
        msg = diff_report(got.data(), want.data())
        assert not msg, f"call, rule {rule}: {msg}"
        # a batch in the buffers of the one before
        s, b = gpu.DeviceSurface(be.ctx, abi.RGBA, W, H), gpu.Batch(be.ctx)
        _leave_edges(lambda *a: b.fill(s, *a))
        b.render(0)
        b.wait()
        b.reset()
        s.upload(init)
        assert b.fill_polygon(s, pat, edges, list(ext), *args) == 0
        b.render(0)
        b.wait()
        out = np.zeros(s.nbytes, np.uint8)
        s.download(out)
        msg = diff_report(out, want.data())
        assert not msg, f"batch, rule {rule}: {msg}"
        b.close()
        s.close()
