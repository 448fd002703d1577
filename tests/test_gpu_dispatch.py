"""How strips reach the two renderers: batches whose tile counts lie around
the strip pass's workgroup size (16 tiles) and beyond the count from which
the general renderer's workgroups take several strips, with strips of both
renderers among them, in the single launch, per surface and longest first:
every surface equals the oracle's, and the work counts are the same."""
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
    from z2d_amd import gpu
    ctx = gpu_backend().ctx
    spec = _spec(n_surfaces, w, h, slow_every, 0xD15 + n_surfaces + w)
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
