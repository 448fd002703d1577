"""Painter calls one after another on one context, which keeps the buffers of
the call before: small after large and large after small, strokes and
polygons between fills, calls that fail between calls that succeed, a call
whose buffers are too large to keep, and calls from two threads at once; each
equal to the oracle's."""
import ctypes as C
import mmap
import threading

import numpy as np
import pytest

from z2d_amd import abi, gpu, scenes
from gpu_util import diff_report, gpu_backend
from oracle_backend import OracleBackend, lib as oracle_lib
from stroke_check import StrokeCheckBackend
from zscene import Surface

pytestmark = pytest.mark.gpu


def _calls(seed, n):
    rng = scenes.SplitMix64(seed)
    out = []
    for i in range(n):
        w, h = rng.randint(1, 300), rng.randint(1, 120)
        if i % 3 == 1:
            w, h = rng.randint(1, 9), rng.randint(1, 9)
        jobs, keep = scenes.random_jobs(rng, 2, w, h, max_side=float(max(4, w)), stroke_share=0.4)
        out.append((w, h, jobs, keep))
    return out


def _run(calls, backend, check):
    for w, h, jobs, _ in calls:
        got, want = Surface(abi.RGBA, w, h), Surface(abi.RGBA, w, h)
        for kind, pat, nodes, opts in jobs:
            assert getattr(backend, kind)(got, pat, nodes, opts) == 0
            assert getattr(check, kind)(want, pat, nodes, opts) == 0
            if kind == "stroke":  # and its outline as a polygon
                rc, edges, ext, aa = gpu.stroke_polygon(nodes, opts, abi.RGBA)
                args = (C.byref(pat), edges.ctypes.data, len(edges), (C.c_double * 4)(*ext), aa,
                        abi.EVEN_ODD, opts.op, opts.precision)
                dg, dw = got.desc(), want.desc()
                assert rc == 0
                assert gpu.lib().z2d_gpu_fill_polygon(backend.ctx.h, C.byref(dg), *args) == 0
                assert oracle_lib().zo_fill_polygon(C.byref(dw), *args) == 0
            bad = nodes.copy()
            bad["tag"][0] = abi.LINE_TO  # a line before any move
            assert backend.fill(got, pat, bad, abi.fill_opts()) != 0
        msg = diff_report(got.data(), want.data())
        assert not msg, f"{w}x{h}: {msg}"


def test_sequence():
    _run(_calls(0x5E9, 24), gpu_backend(), StrokeCheckBackend())


def test_large_call_between_small_ones():
    be, ob = gpu_backend(), OracleBackend()
    rng = scenes.SplitMix64(0x1A6)
    # a polyline of 20,000 lines down a tall surface: some 3.4 million (edge,
    # band) copies of 32 bytes, beyond the 64 MiB that a context keeps
    n, w, h = 20000, 64, 8192
    pts = [(rng.uniform(0, w), rng.uniform(0, h)) for _ in range(n)]
    big = abi.nodes_array([(abi.MOVE_TO, *pts[0])] + [(abi.LINE_TO, *p) for p in pts[1:]] +
                          [(abi.CLOSE_PATH,), (abi.MOVE_TO, *pts[0])])
    pat = abi.solid_pattern(abi.rgba(10, 60, 90, 100))
    small = scenes.star_512()["draws"][0]
    for nodes, sw, sh in ((small[1], 80, 512), (big, w, 64), (small[1], 80, 512), (big, w, h),
                          (small[1], 512, 80)):
        got, want = Surface(abi.RGBA, sw, sh), Surface(abi.RGBA, sw, sh)
        opts = abi.fill_opts(abi.AA_DEFAULT, abi.EVEN_ODD, "src_over")
        assert be.fill(got, pat, nodes, opts) == 0
        assert ob.fill(want, pat, nodes, opts) == 0
        msg = diff_report(got.data(), want.data())
        assert not msg, f"{sw}x{sh}: {msg}"


def _resident():
    with open("/proc/self/statm") as f:
        return int(f.read().split()[1]) * mmap.PAGESIZE


def test_inputs_of_a_failed_call_are_not_kept():
    """8.6 million edges down 512 bands are more (edge, band) pairs than a
    batch can index, which is found before any buffer is made: the context
    keeps none of the 275 MB either."""
    be, s = gpu_backend(), Surface(abi.RGBA, 64, 8192)
    edges = np.zeros(8600000, abi.EDGE_DTYPE)
    edges["y1"] = 4.0 * 8192
    d, pat = s.desc(), abi.solid_pattern(abi.rgba(1, 2, 3, 4))
    ext = (C.c_double * 4)(0.0, 4.0 * 8192, 0.0, 256.0)
    before = _resident()
    assert gpu.lib().z2d_gpu_fill_polygon(be.ctx.h, C.byref(d), C.byref(pat), edges.ctypes.data,
                                          len(edges), ext, abi.AA_DEFAULT, 0, abi.OP["src_over"],
                                          0) == abi.ERR_OUT_OF_MEMORY
    assert _resident() - before < 128 << 20
    _run(_calls(0xF41, 2), be, StrokeCheckBackend())


def test_two_threads():
    be = gpu_backend()
    errs = []

    def work(seed):
        try:
            _run(_calls(seed, 10), be, StrokeCheckBackend())
        except BaseException as e:  # noqa: BLE001
            errs.append(e)

    th = [threading.Thread(target=work, args=(0x71 + k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
