"""Multisampled src of a solid paint and clear, the draws that replace what
they cover, between src_over draws, over every format and both precisions:
equal to the oracle (an opaque format stays opaque, packed alpha keeps its
bits, uncovered pixels their value)."""
import numpy as np
import pytest

from z2d_amd import abi, scenes
from gpu_util import diff_report, gpu_backend, run_draws
from oracle_backend import OracleBackend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", list(range(8)), ids=abi.FORMAT_NAMES)
@pytest.mark.parametrize("prec", [0, 1], ids=["int", "float"])
def test_replace(fmt, prec):
    w, h = 150, 37
    rng = scenes.SplitMix64(0x4E9 + fmt + 8 * prec)
    draws, keep = [], []
    for i in range(12):
        op = ("src_over", "src", "clear", "src_over", "src", "src_over")[i % 6]
        d, k = scenes.random_paths(rng, 1, w, h, max_side=120.0, gradients=op != "src", op=op)
        pat, nodes, opts = d[0]
        opts.precision = prec if op != "src_over" else 0
        if i == 4:
            pat = abi.solid_pattern(abi.pixel(abi.ALPHA8, a=90))
        draws.append((pat, nodes, opts))
        keep.append(k)
    init = rng.u8_array(abi.surface_nbytes(fmt, w, h))
    if fmt in (abi.RGBA, abi.ARGB):
        init = scenes.premultiplied_rgba(fmt + 5, w * h)
    if fmt in (abi.RGB, abi.XRGB):
        init.reshape(-1, 4)[:, 3] = 0
    want = run_draws(OracleBackend(), fmt, w, h, init, draws)
    got = run_draws(gpu_backend(), fmt, w, h, init, draws)
    msg = diff_report(got.data(), want.data())
    assert not msg, msg
