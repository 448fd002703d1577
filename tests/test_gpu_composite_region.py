"""Regions of the per-operator compositor: rows of every length modulo four
(the last quad of a row), narrower and wider than a workgroup's row of lanes,
offsets that put rows at every address modulo 16, sources larger than the
region, and whole surfaces whose pixel count is not a multiple of four, on
host and device surfaces: equal to the oracle, and nothing written beside
the region."""
import ctypes as C

import numpy as np
import pytest

from z2d_amd import abi
from z2d_amd.scenes import SplitMix64
from gpu_util import diff_report, gpu_backend
from oracle_backend import OracleBackend
from test_gpu_composite import rand_surface

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y,sw,sh", [(0, 0, 7, 3), (1, 0, 5, 4), (2, 1, 4, 9), (3, 2, 9, 1),
                                       (-3, -1, 20, 6), (5, 3, 1, 5), (7, 0, 263, 5),
                                       (-2, 0, 300, 70), (0, 0, 271, 68), (0, 0, 271, 80),
                                       (270, 67, 3, 3)])
@pytest.mark.parametrize("op", ["src", "src_over", "overlay", "soft_light"])
def test_regions(x, y, sw, sh, op):
    w, h = 271, 68
    rng = SplitMix64(0x9E6 + 31 * sw + sh + x)
    for fmt, masked in ((abi.RGBA, False), (abi.XRGB, True)):
        dst = rand_surface(rng, fmt, w, h)
        src = rand_surface(rng, abi.ARGB, max(sw, w) if masked else sw, max(sh, h) if masked else sh)
        sd = src.desc()
        o = abi.CompOp()
        o.op = abi.OP[op]
        ops, keep = [o], [sd]
        if masked:  # the masked source is read at the destination, the mask from its start
            mask = rand_surface(rng, abi.ALPHA8, sw, sh)
            md = mask.desc()
            m = abi.CompOp()
            m.op = abi.OP["dst_in"]
            m.dst.kind = m.src.kind = abi.PARAM_SURFACE
            m.dst.surface, m.src.surface = C.pointer(sd), C.pointer(md)
            ops = [m, o]
            keep += [mask, md]
        else:
            o.src.kind = abi.PARAM_SURFACE
            o.src.surface = C.pointer(sd)
        want, got = dst.copy(), dst.copy()
        assert OracleBackend().composite(want, x, y, ops, 0) == 0
        assert gpu_backend().composite(got, x, y, ops, 0) == 0
        msg = diff_report(got.data(), want.data())
        assert not msg, f"fmt {fmt} masked {masked}: {msg}"


@pytest.mark.parametrize("w,h", [(1, 1), (1, 3), (3, 1), (33, 31), (1025, 3)])
def test_device_surfaces_out_of_place(w, h):
    from z2d_amd import gpu
    ctx = gpu_backend().ctx
    rng = SplitMix64(0x0DD + w * h)
    dst, src = rand_surface(rng, abi.RGBA, w, h), rand_surface(rng, abi.RGBA, w, h)
    want = dst.copy()
    sd = src.desc()
    o = abi.CompOp()
    o.op = abi.OP["xor"]
    o.src.kind = abi.PARAM_SURFACE
    o.src.surface = C.pointer(sd)
    assert OracleBackend().composite(want, 0, 0, [o], 0) == 0
    devs = [gpu.DeviceSurface(ctx, abi.RGBA, w, h) for _ in range(3)]
    for d, s in zip(devs, (dst, src)):
        d.upload(s.buf[: d.nbytes].copy())
    ds = devs[1].desc()
    o.src.surface = C.pointer(ds)
    dd, do = devs[0].desc(), devs[2].desc()
    for f in (gpu.lib().z2d_gpu_composite, gpu.lib().z2d_gpu_composite_noalloc):
        ctx.check(f(ctx.h, C.byref(dd), 0, 0, (abi.CompOp * 1)(o), 1, 0, C.byref(do)), "composite")
        got = np.zeros(devs[2].nbytes, np.uint8)
        devs[2].download(got)
        msg = diff_report(got, want.data())
        assert not msg, msg
    for d in devs:
        d.close()
