"""How strips reach the two renderers: batches whose tile counts lie around
the strip pass's workgroup size (16 tiles), with strips of both renderers
among them, and beyond the counts from which the general renderer's workgroups
take several strips (more than 8,192 of its strips) and the list passes' waves
several tiles (more than 8,192) or slots; in the single launch, per surface
and longest first: every surface equals the oracle's, and the work counts are
the same."""
import numpy as np
import pytest

from z2d_amd import abi, scenes
from gpu_util import diff_report, gpu_backend
from oracle_backend import OracleBackend
from zscene import Surface

pytestmark = pytest.mark.gpu


def _spec(n_surfaces, w, h, slow_every, seed):
    rng = scenes.SplitMix64(seed)
    spec = []
    for i in range(n_surfaces):
        draws, keep = scenes.random_paths(rng, 2, w, h, max_side=float(min(w, h)))
        if slow_every and i % slow_every == 0:  # an operator of the general renderer
            more, k = scenes.random_paths(rng, 1, w, h, max_side=float(min(w, h)), op="multiply")
            draws, keep = draws + more, keep + k
        spec.append((draws, keep))
    return spec


@pytest.mark.parametrize("n_surfaces,w,h,slow_every",
                         [(1, 60, 5, 0), (1, 60, 5, 1), (15, 64, 16, 2), (16, 64, 16, 1),
                          (17, 64, 16, 16), (5, 130, 33, 2), (2, 1500, 1500, 2)])
def test_strips_of_both_renderers(n_surfaces, w, h, slow_every):
    _check(_spec(n_surfaces, w, h, slow_every, 0xD15 + n_surfaces + w), w, h)


def _whole(w, h, op):
    """A rectangle over the whole surface."""
    nodes = abi.nodes_array([(abi.MOVE_TO, 0.0, 0.0), (abi.LINE_TO, w, 0.0), (abi.LINE_TO, w, h),
                             (abi.LINE_TO, 0.0, h), (abi.CLOSE_PATH,), (abi.MOVE_TO, 0.0, 0.0)])
    return (abi.solid_pattern(abi.rgba(200, 150, 220, 240)), nodes,
            abi.fill_opts(abi.AA_DEFAULT, abi.NON_ZERO, op))


def test_workgroups_of_several_strips():
    """10,200 tiles; 20,400 of the 40,800 strips are the general renderer's,
    which gets 10,200 workgroups, each of which finds the LDS of the strip
    before (the multiply's rows after a denser draw's)."""
    w, h = 1600, 1632
    spec = _spec(4, w, h, 0, 0x5E7)
    for i in (1, 2):
        spec[i] = ([_whole(w, h, "src_over")] + spec[i][0] + [_whole(w, h, "multiply")], spec[i][1])
    _check(spec, w, h)


def test_slots_of_many_draws():
    """256 bands and 36 groups of 64 draws: 9,216 slots."""
    w, h = 64, 4096
    rng = scenes.SplitMix64(0x510)
    draws, keep = scenes.random_paths(rng, 2300, w, h, max_side=40.0)
    _check([(draws, keep)], w, h)


def _check(spec, w, h):
    from z2d_amd import gpu
    ctx = gpu_backend().ctx
    want = []
    for draws, _ in spec:
        s = Surface(abi.RGBA, w, h)
        for pat, nodes, opts in draws:
            assert OracleBackend().fill(s, pat, nodes, opts) == 0
        want.append(s.data())
    counts = {}
    for mode, longest in ((0, 0), (1, 0), (0, 1)):
        b = gpu.Batch(ctx)
        surfs = []
        for draws, _ in spec:
            s = gpu.DeviceSurface(ctx, abi.RGBA, w, h)
            surfs.append(s)
            for pat, nodes, opts in draws:
                assert b.fill(s, pat, nodes, opts) == 0
        b.set_queue_order(longest)
        b.prepare()
        b.counters(True)
        b.render(mode)
        b.wait()
        counts[(mode, longest)] = b.counters(False)[:5]
        for i, s in enumerate(surfs):
            got = np.zeros(s.nbytes, np.uint8)
            s.download(got)
            msg = diff_report(got, want[i])
            assert not msg, f"mode {mode} longest {longest} surface {i}: {msg}"
        b.render(mode)  # without counting
        b.wait()
        assert b.counters(False)[0] == 0
        b.close()
        for s in surfs:
            s.close()
    assert len(set(counts.values())) == 1 and counts[(0, 0)][0] > 0, counts
