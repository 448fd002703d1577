"""Whole surfaces painted with gradients and dithers (the compositor's paint
kernel and, past its limits, the general one): every gradient type, 1 to 9
stops with hard ones among them, the dither types over a gradient and a
color, widths of every remainder of four and beyond a lane's step, several
operators and formats: equal to the oracle."""
import ctypes as C

import numpy as np
import pytest

from z2d_amd import abi
from z2d_amd.scenes import SplitMix64, rgba_from_clamped
from gpu_util import diff_report, gpu_backend
from oracle_backend import OracleBackend
from test_gpu_composite import rand_surface

pytestmark = pytest.mark.gpu


def _gradient(rng, gtype, n, w, h):
    geom = ([rng.uniform(0, w), rng.uniform(0, h), rng.uniform(0, w), rng.uniform(0, h)],
            [rng.uniform(0, w), rng.uniform(0, h), 3.0, rng.uniform(0, w), rng.uniform(0, h), w / 2.0],
            [rng.uniform(0, w), rng.uniform(0, h), rng.uniform(0, 6.3)])[gtype]
    offs = sorted(rng.uniform() for _ in range(n))
    if n > 3:
        offs[2] = offs[1]  # a hard stop
    stops = [(o, abi.color(abi.COLOR_LINEAR_RGB, rng.uniform(), rng.uniform(), rng.uniform(),
                           0.0 if i == 3 else rng.uniform())) for i, o in enumerate(offs)]
    m = abi.IDENTITY if rng.uniform() < 0.5 else (0.8, 0.3, -0.2, 1.1, 2.0, -1.0)
    return abi.Gradient(gtype, geom, stops, abi.INTERP_LINEAR_RGB, matrix=m)


@pytest.mark.parametrize("gtype", [0, 1, 2])
@pytest.mark.parametrize("n,w,h", [(1, 1, 1), (2, 5, 3), (4, 6, 9), (5, 63, 5), (8, 259, 7),
                                   (9, 40, 6), (3, 1030, 2)])
@pytest.mark.parametrize("dither", [None, 0, 1, 2])
def test_gradient(gtype, n, w, h, dither):
    rng = SplitMix64(0x9A17 + gtype + 7 * n + w)
    for fmt, op in ((abi.RGBA, "src"), (abi.ARGB, "src_over"), (abi.XRGB, "multiply")):
        dst = rand_surface(rng, fmt, w, h)
        g = _gradient(rng, gtype, n, w, h)
        o = abi.CompOp()
        o.op = abi.OP[op]
        if dither is None:
            o.src.kind = abi.PARAM_GRADIENT
            o.src.gradient = C.pointer(g.desc)
        else:
            o.src.kind = abi.PARAM_DITHER
            o.src.dither = abi.dither_pattern(dither, rng.randint(1, 8), gradient=g).dither
        want, got = dst.copy(), dst.copy()
        assert OracleBackend().composite(want, 0, 0, [o], 0) == 0
        assert gpu_backend().composite(got, 0, 0, [o], 0) == 0
        msg = diff_report(got.data(), want.data())
        assert not msg, f"{fmt} {op}: {msg}"


@pytest.mark.parametrize("gtype", [0, 1, 2])
@pytest.mark.parametrize("w,h", [(1024, 320), (1025, 320), (5003, 67)])
@pytest.mark.parametrize("dither", [None, 2])
def test_lane_of_one_and_of_four_pixels(gtype, w, h, dither):
    """327,680 pixels are the most that are painted by a lane each; beyond,
    a lane's four, and a row of more than 16 workgroups' in several steps."""
    test_gradient(gtype, 6, w, h, dither)


@pytest.mark.parametrize("dither", [0, 1, 2])
def test_color_dither(dither):
    rng = SplitMix64(0xC01 + dither)
    for fmt, op, w, h in ((abi.RGBA, "src", 67, 66), (abi.RGB, "src_over", 130, 5)):
        dst = rand_surface(rng, fmt, w, h)
        for col in (None, abi.color(abi.COLOR_SRGB, 0.2, 0.7, 0.4, 0.6)):
            px = rgba_from_clamped(rng.uniform(), rng.uniform(), rng.uniform(), 0.8)
            o = abi.CompOp()
            o.op = abi.OP[op]
            o.src.kind = abi.PARAM_DITHER
            o.src.dither = abi.dither_pattern(dither, 4, px=None if col else px, col=col).dither
            want, got = dst.copy(), dst.copy()
            assert OracleBackend().composite(want, 0, 0, [o], 0) == 0
            assert gpu_backend().composite(got, 0, 0, [o], 0) == 0
            msg = diff_report(got.data(), want.data())
            assert not msg, f"{fmt} {op}: {msg}"
