"""Calls of one context on several streams and in HIP graphs: what the workgroup
schedule's launches keep in the context must not reach another launch that is
still running, nor a graph that is replayed later."""
import ctypes as C

import numpy as np
import pytest

from onekapy_amd import _lib
from onekapy_amd.sites import fixed_field
from helpers import oracle_fit_draw, small_site
from test_zz_no_alloc import DeviceSite, HipMemory

pytestmark = pytest.mark.gpu

PRECISIONS = pytest.mark.parametrize("precision", [_lib.FP64_EXACT, _lib.FP32],
                                     ids=["fp64", "fp32"])


class Launches:
    """Asynchronous launches of device-resident sites, on streams of their own."""

    def __init__(self):
        self.mem, self.ctx = HipMemory(), _lib.context()
        self.hip = self.mem.hip
        self.streams = []
        for f, args in (("hipStreamCreateWithFlags", [C.POINTER(C.c_void_p), C.c_uint]),
                        ("hipStreamSynchronize", [C.c_void_p]),
                        ("hipStreamDestroy", [C.c_void_p]),
                        ("hipStreamBeginCapture", [C.c_void_p, C.c_int]),
                        ("hipStreamEndCapture", [C.c_void_p, C.POINTER(C.c_void_p)]),
                        ("hipGraphInstantiate", [C.POINTER(C.c_void_p), C.c_void_p, C.c_void_p,
                                                 C.c_void_p, C.c_size_t]),
                        ("hipGraphLaunch", [C.c_void_p, C.c_void_p]),
                        ("hipGraphExecDestroy", [C.c_void_p]),
                        ("hipGraphDestroy", [C.c_void_p])):
            getattr(self.hip, f).argtypes = args

    def do(self, name, *args):
        assert getattr(self.hip, name)(*args) == 0, name

    def stream(self):
        s = C.c_void_p()
        self.do("hipStreamCreateWithFlags", C.byref(s), 1)
        self.streams.append(s)
        return s

    def site(self, seed, nreal, npaths, spacing, nside):
        s, d = small_site(nreal=nreal, npaths=npaths, seed=seed)
        if seed % 2:   # other places about the target: another field
            s.wells = [w if i == s.target else (w[0] + 37.0, w[1] - 21.0) + tuple(w[2:])
                       for i, w in enumerate(s.wells)]
        _, _, coef = oracle_fit_draw(s, d)
        pf = fixed_field(s.xt, s.yt, spacing, nside, nside)
        ds = DeviceSite(self.mem, s, d, coef, pf, s.umbra, npaths)
        ds.nreal, ds.shape = nreal, (nside, nside)
        g = ds.grid
        ds.epoch = self.mem.put(np.frombuffer(bytes(_lib.Epoch_(0, g.xmin, g.ymin, g.nrows,
                                                                g.ncols, 0, 0)), np.uint8))
        ds.counts = self.mem.put(np.zeros(ds.shape, np.int32))
        return ds

    def launch(self, ds, precision, flags=_lib.PTR_DEVICE | _lib.ASYNC, **kw):
        opts = _lib.make_trace_opts(ds.P, ds.s.duration, ds.s.tol, ds.s.maxstep, ds.umbra,
                                    ds.starts, precision, True,
                                    schedule=_lib.SCHED_WORKGROUP, **kw)
        self.ctx.check(self.ctx.lib.oka_trace_chronicle(
            self.ctx.h, C.byref(ds.site), ds.nreal, ds.K, ds.n, ds.b, ds.q, ds.coef,
            C.byref(opts), C.byref(ds.grid), 1, ds.epoch, 1, ds.counts, None, None, None, None,
            flags))

    def clear(self, ds):
        zeros = np.zeros(ds.shape, np.int32)
        self.do("hipMemcpy", ds.counts, zeros.ctypes.data, zeros.nbytes, HipMemory.H2D)

    def counts(self, ds):
        return self.mem.get(ds.counts, ds.shape, np.int32)

    def alone(self, ds, precision, **kw):
        """The counts of a synchronous launch with nothing else running."""
        self.launch(ds, precision, _lib.PTR_DEVICE, **kw)
        out = self.counts(ds)
        self.clear(ds)
        assert out.any()
        return out

    def close(self):
        self.ctx.set_stream(None)
        for s in self.streams:
            self.do("hipStreamSynchronize", s)
            self.do("hipStreamDestroy", s)
        self.mem.close()


@pytest.fixture
def launches(gpu_ctx):
    run = Launches()
    yield run
    run.close()


@PRECISIONS
def test_overlapping_launches_on_streams_of_one_context(launches, precision):
    """Two sites in turn on three streams, six launches in flight, more than a
    workgroup's lanes of particles each: the counts of each alone."""
    sites = [launches.site(k, 1500 - 400 * k, 300 + 100 * k, 40.0, 100) for k in (0, 1)]
    want = [launches.alone(ds, precision) for ds in sites]
    streams = [launches.stream() for _ in range(3)]
    for k in range(6):
        launches.ctx.set_stream(streams[k % 3])
        launches.launch(sites[k % 2], precision)
    for s in streams:
        launches.do("hipStreamSynchronize", s)
    for ds, w in zip(sites, want):
        assert np.array_equal(launches.counts(ds), 3 * w)


@PRECISIONS
def test_captured_launch_outlives_larger_calls(launches, precision):
    """A captured launch, replayed after calls with another site, more
    realizations and a larger grid have used (and grown) the context's
    buffers, and while one of them runs."""
    ds = launches.site(0, 700, 400, 40.0, 100)
    big = launches.site(1, 2600, 300, 10.0, 500)
    want, want_big = launches.alone(ds, precision), launches.alone(big, precision)
    s, s2 = launches.stream(), launches.stream()
    launches.ctx.set_stream(s)
    graph, ex = C.c_void_p(), C.c_void_p()
    launches.do("hipStreamBeginCapture", s, 2)   # relaxed
    launches.launch(ds, precision)
    launches.do("hipStreamEndCapture", s, C.byref(graph))
    launches.do("hipGraphInstantiate", C.byref(ex), graph, None, None, 0)
    launches.ctx.set_stream(s2)
    for k in range(4):
        if k > 0:
            launches.launch(big, precision)
        launches.do("hipGraphLaunch", ex, s)
        if k == 2:
            launches.launch(big, precision)
        launches.do("hipStreamSynchronize", s)
        launches.do("hipStreamSynchronize", s2)
        assert np.array_equal(launches.counts(ds), want), k
        launches.clear(ds)
        n = (k > 0) + (k == 2)
        assert np.array_equal(launches.counts(big), n * want_big), k
        launches.clear(big)
    launches.do("hipGraphExecDestroy", ex)
    launches.do("hipGraphDestroy", graph)


@PRECISIONS
def test_captured_launch_needs_no_more_memory_than_its_warm_up(launches, precision):
    """Bitmaps in HBM, more realizations than workgroups at once: the regions of
    the captured launch are no larger than those of the eager one before it."""
    ds = launches.site(0, 2500, 260, 40.0, 100)
    want = launches.alone(ds, precision, bitmap_mode=_lib.BITMAP_HBM_FLAT)
    s = launches.stream()
    launches.ctx.set_stream(s)
    graph, ex = C.c_void_p(), C.c_void_p()
    launches.do("hipStreamBeginCapture", s, 2)   # relaxed
    launches.launch(ds, precision, bitmap_mode=_lib.BITMAP_HBM_FLAT)
    launches.do("hipStreamEndCapture", s, C.byref(graph))
    launches.do("hipGraphInstantiate", C.byref(ex), graph, None, None, 0)
    for k in range(3):
        launches.do("hipGraphLaunch", ex, s)
        launches.do("hipStreamSynchronize", s)
        assert np.array_equal(launches.counts(ds), want), k
        launches.clear(ds)
    launches.do("hipGraphExecDestroy", ex)
    launches.do("hipGraphDestroy", graph)
