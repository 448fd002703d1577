"""The fast strip worker's crossing words at the windings where their layout
changes: closed paths that go round 1 to 300 times in either direction (a
byte holds windings to 127, 254 edges are the most that cannot exceed it),
slanted so that the loops cross several strips and lie left of others, both
fill rules, and the same between hundreds of short edges, where a strip's
edges are many but a sample row's crossings few; equal to the oracle."""
import math

import numpy as np
import pytest

from z2d_amd import abi
from gpu_util import diff_report, gpu_backend, run_draws
from oracle_backend import OracleBackend

pytestmark = pytest.mark.gpu


def _loops(n, sign, w, h, twist):
    """n rounds of a slanted quadrilateral, its corners drifting by `twist`."""
    base = [(9.3, 1.7), (w - 70.4, 2.2), (w - 11.1, h - 2.6), (33.8, h - 1.1)]
    if sign < 0:
        base = base[::-1]
    pts = [(x + twist * i, y) for i in range(n) for x, y in base]
    nodes = [(abi.MOVE_TO, *pts[0])] + [(abi.LINE_TO, *p) for p in pts[1:]]
    return abi.nodes_array(nodes + [(abi.CLOSE_PATH,), (abi.MOVE_TO, *pts[0])])


@pytest.mark.parametrize("rule", [abi.NON_ZERO, abi.EVEN_ODD])
@pytest.mark.parametrize("n", [1, 2, 63, 126, 127, 128, 129, 300])
def test_loops(n, rule):
    w, h = 230, 21
    init = (np.arange(w * h * 4, dtype=np.uint32) * 2654435761 >> 24).astype(np.uint8)
    init = init.reshape(-1, 4)
    init[:, :3] = np.minimum(init[:, :3], init[:, 3:])
    draws = []
    for sign, twist in ((1, 0.0), (-1, 0.0), (1, 0.037), (-1, -0.021)):
        # a translucent paint, so that wrong coverage in any draw shows
        draws.append((abi.solid_pattern(abi.rgba(40, 90, 20, 120)), _loops(n, sign, w, h, twist),
                      abi.fill_opts(abi.AA_DEFAULT, rule, "src_over")))
    want = run_draws(OracleBackend(), abi.RGBA, w, h, init.reshape(-1), draws)
    got = run_draws(gpu_backend(), abi.RGBA, w, h, init.reshape(-1), draws)
    msg = diff_report(got.data(), want.data())
    assert not msg, msg


@pytest.mark.parametrize("n", [0, 1, 30, 62, 63, 64, 65, 100])
def test_loops_among_short_edges(n):
    """2n crossings of a sample row by the loops, and those of two wavy
    columns of 500 short edges each (a stroke's outline looks like that)."""
    w, h = 230, 21
    init = np.full(w * h * 4, 255, np.uint8)
    draws = []
    for sign, twist, x0 in ((1, 0.0, 20.0), (-1, 0.03, 100.0), (1, -0.02, 215.0)):
        loops = _loops(max(1, n), sign, w, h, twist)[:-1] if n else np.zeros(0, abi.NODE_DTYPE)
        m = 500
        side = [(x0 + 3.0 * math.sin(0.7 * i), 1.0 + (h - 2.0) * i / m) for i in range(m + 1)]
        pts = side + [(x + 6.0, y) for x, y in side[::-1]]
        wavy = abi.nodes_array([(abi.MOVE_TO, *pts[0])] + [(abi.LINE_TO, *p) for p in pts[1:]] +
                               [(abi.CLOSE_PATH,), (abi.MOVE_TO, *pts[0])])
        draws.append((abi.solid_pattern(abi.rgba(40, 90, 20, 120)), np.concatenate([loops, wavy]),
                      abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, "src_over")))
    want = run_draws(OracleBackend(), abi.RGBA, w, h, init, draws)
    got = run_draws(gpu_backend(), abi.RGBA, w, h, init, draws)
    msg = diff_report(got.data(), want.data())
    assert not msg, msg
