"""Edges built 64 node slots at a time: draws whose contours start, close and
end around the groups' borders (closes first and last in a group, contours of
one to three points, closes on their first point, runs of closes, a line or a
curve after a close), and few and many edges against few and many bands
(surfaces of 1 to 132 bands of 16 rows, other band heights), equal to the
oracle."""
import numpy as np
import pytest

from z2d_amd import abi, scenes
from gpu_util import diff_report, gpu_backend, run_draws
from oracle_backend import OracleBackend
from zscene import Surface

pytestmark = pytest.mark.gpu


def _path(rng, n_target, w, h, kinds):
    """Contours until n_target nodes; kinds: weights of what a contour is."""
    nodes = []
    while len(nodes) < n_target:
        k = kinds[rng.randint(0, len(kinds) - 1)]
        p0 = (rng.uniform(-5, w + 5), rng.uniform(-5, h + 5))
        nodes.append((abi.MOVE_TO, *p0))
        m = {"short": rng.randint(0, 2), "poly": rng.randint(3, 40)}.get(k, rng.randint(2, 6))
        last = p0
        for _ in range(m):
            last = (rng.uniform(-5, w + 5), rng.uniform(-5, h + 5))
            nodes.append((abi.LINE_TO, *last))
            if rng.uniform() < 0.1:
                nodes.append((abi.LINE_TO, *last))  # a line that does not move
        if k == "back":
            nodes.append((abi.LINE_TO, *p0))  # closes on its first point
        nodes.append((abi.CLOSE_PATH,))
        if k == "runs":
            nodes += [(abi.CLOSE_PATH,)] * rng.randint(1, 3)
        if k == "after":
            nodes.append((abi.LINE_TO, rng.uniform(0, w), rng.uniform(0, h)))
            nodes.append((abi.CURVE_TO, *[rng.uniform(0, w) for _ in range(6)]))
            nodes.append((abi.CLOSE_PATH,))
    return abi.nodes_array(nodes + [(abi.MOVE_TO, *p0)])


@pytest.mark.parametrize("kinds", [("poly", "back"), ("short", "poly", "back", "runs"),
                                   ("poly", "after", "short")], ids=["plain", "odd", "after"])
@pytest.mark.parametrize("n", [3, 62, 63, 64, 65, 127, 129, 200, 700])
def test_group_borders(n, kinds):
    w, h = 90, 70
    rng = scenes.SplitMix64(0xE6 + n * 7 + len(kinds))
    draws = []
    for rule, aa in ((abi.EVEN_ODD, abi.AA_DEFAULT), (abi.NON_ZERO, abi.AA_DEFAULT),
                     (abi.NON_ZERO, abi.AA_NONE)):
        draws.append((abi.solid_pattern(abi.rgba(60, 20, 90, 110)), _path(rng, n, w, h, kinds),
                      abi.fill_opts(aa, rule, "src_over")))
    init = np.full(w * h * 4, 255, np.uint8)
    want = run_draws(OracleBackend(), abi.RGBA, w, h, init, draws)
    got = run_draws(gpu_backend(), abi.RGBA, w, h, init, draws)
    msg = diff_report(got.data(), want.data())
    assert not msg, msg


@pytest.mark.parametrize("band", [4, 16, 32])
@pytest.mark.parametrize("w,h", [(40, 3), (33, 16), (20, 1025), (24, 2110)])
def test_edges_and_bands(w, h, band):
    from z2d_amd import gpu
    ctx = gpu_backend().ctx
    rng = scenes.SplitMix64(0xBA0D + w + h)
    rect = abi.nodes_array([(abi.MOVE_TO, 1.5, -3.0), (abi.LINE_TO, w - 2.25, -3.0),
                            (abi.LINE_TO, w - 1.0, h + 9.0), (abi.LINE_TO, 0.5, h - 0.4),
                            (abi.CLOSE_PATH,), (abi.MOVE_TO, 1.5, -3.0)])
    paths = [rect] + [_path(rng, n, w, h, ("poly", "back")) for n in (12, 60, 90, 300)]
    pat = abi.solid_pattern(abi.rgba(30, 70, 10, 90))
    want, surf, b = Surface(abi.RGBA, w, h), gpu.DeviceSurface(ctx, abi.RGBA, w, h), gpu.Batch(ctx)
    for i, p in enumerate(paths):
        opts = abi.fill_opts(abi.AA_DEFAULT, i & 1, "src_over")
        assert OracleBackend().fill(want, pat, p, opts) == 0
        assert b.fill(surf, pat, p, opts) == 0
    b.set_band_height(band)
    got = np.zeros(surf.nbytes, np.uint8)
    for _ in range(2):  # the second render starts from the first one's leftovers
        surf.upload(np.zeros(surf.nbytes, np.uint8))
        b.render(0)
        b.wait()
        surf.download(got)
        msg = diff_report(got, want.data())
        assert not msg, msg
    b.close()
    surf.close()
