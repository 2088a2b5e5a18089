"""Calls of one handle on several streams, unchecked, so that nothing waits on the host
between them: the binned calls share the handle's work space and its derived tables, and each
must still get exactly what it gets alone.  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from test_gpu_small_calls import device_call, points

pytestmark = pytest.mark.gpu


class Stream:
    def __init__(self):
        self.p = C.c_void_p()
        capi.check(capi.lib().brille_stream_create(C.byref(self.p)))

    def __del__(self):
        capi.lib().brille_stream_destroy(self.p)


class Call:
    """Q and outputs in device memory, allocated beforehand."""

    def __init__(self, dev, Q, precision):
        vs, cs = dev.out_shapes(len(Q))
        f32 = precision == capi.FP32
        self.dev, self.n, self.precision = dev, len(Q), precision
        self.Q = capi.DeviceArray.from_host(Q)
        self.out = (capi.DeviceArray(vs, np.float32 if f32 else np.float64),
                    capi.DeviceArray(cs, np.complex64 if f32 else np.complex128))

    def run(self, stream, kernel, entry="brille_ir_interpolate_at", check=0):
        o = capi.RunOpts(0, self.precision, 0, capi.MEM_DEVICE, kernel, check)
        capi.check(getattr(capi.lib(), entry)(self.dev.h, self.Q.ptr, self.n, C.byref(o), self.out[0].ptr,
                                              self.out[1].ptr, None, stream.p if stream else None))


def grid_tables(spec, v_target=600.0):
    sp = dict(S.batch_specs(16)[spec], v_target=v_target)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    return g, dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)


# 4 and 24 atoms; sizes AUTO gives to the pipeline
# (every seventh call is checked: the host waits for it, and the next ones need not)
@pytest.mark.parametrize("spec,precision,sizes,kernel", [
    (7, capi.FP64, (60_000, 75_000), capi.KERNEL_AUTO), (7, capi.FP32, (120_000, 100_000), capi.KERNEL_AUTO),
    (5, capi.FP64, (2_000, 3_000), capi.KERNEL_AUTO), (3, capi.FP32, (50_000, 400_000), capi.KERNEL_BINNED)])
def test_unchecked_calls_on_two_streams_and_the_null_stream(spec, precision, sizes, kernel):
    print(f"streams: grid {spec} {precision} {sizes}", flush=True)
    g, t = grid_tables(spec)
    r = np.random.default_rng(5)
    Qs = [points(g, r, n) for n in sizes * 3]
    ref = capi.Grid(t)
    want = [[x.to_host() for x in device_call(ref, Q, precision, capi.KERNEL_TILE)[1:]] for Q in Qs]
    for _ in range(3):  # a fresh handle each time: its first call also builds the table
        dev = capi.Grid(t)
        calls = [Call(dev, Q, precision) for Q in Qs]
        streams = [Stream(), Stream(), None]
        capi.check(capi.lib().brille_device_sync())
        for k in range(2 * len(calls)):
            calls[k % len(calls)].run(streams[k % 3], kernel, check=int(k % 7 == 3))
        capi.check(capi.lib().brille_device_sync())
        for c, w in zip(calls, want):
            for a, b in zip(c.out, w):
                np.testing.assert_array_equal(a.to_host(), b)


def test_unchecked_allocation_free_calls_of_two_handles():
    """They share one array per GPU, which only large calls work in: two ordinary ones (here with
    their tables built) may run side by side."""
    print("streams: allocation-free calls", flush=True)
    g, t = grid_tables(7)
    r = np.random.default_rng(6)
    devs, streams = [capi.Grid(t), capi.Grid(t)], [Stream(), Stream()]
    Qs = [points(g, r, n) for n in (60_000, 70_000)]
    want = [[x.to_host() for x in device_call(d, Q, capi.FP64, capi.KERNEL_TILE)[1:]] for d, Q in zip(devs, Qs)]
    for d in devs:
        device_call(d, Qs[0], capi.FP64, capi.KERNEL_BINNED)
    calls = [Call(d, Q, capi.FP64) for d, Q in zip(devs, Qs)]
    capi.check(capi.lib().brille_device_sync())
    for _ in range(5):
        for c, s in zip(calls, streams):
            c.run(s, capi.KERNEL_AUTO, "brille_ir_interpolate_at_noalloc")
    capi.check(capi.lib().brille_device_sync())
    for c, w in zip(calls, want):
        for a, b in zip(c.out, w):
            np.testing.assert_array_equal(a.to_host(), b)


def hip_runtime():
    maps = open("/proc/self/maps").read().split()
    return C.CDLL(next(m for m in maps if "libamdhip64" in m))  # the one the library itself uses


class Graph:
    """Calls recorded on a stream of their own (mode 0: global, 1: thread-local)."""

    def __init__(self, mode, record):
        self.hip, self.s, graph = hip_runtime(), Stream(), C.c_void_p()
        self.exec = C.c_void_p()
        capi.check(capi.lib().brille_device_sync())
        assert self.hip.hipStreamBeginCapture(self.s.p, mode) == 0
        try:
            record(self.s)
        finally:
            assert self.hip.hipStreamEndCapture(self.s.p, C.byref(graph)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)) == 0
        assert self.hip.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.s.p) == 0

    def __del__(self):
        self.hip.hipGraphExecDestroy(self.exec)


def clobber(call):
    for x in call.out:
        junk = np.full(x.shape, 7, x.dtype)
        capi.check(capi.lib().brille_memcpy_h2d(x.ptr, junk.ctypes.data_as(C.c_void_p), x.nbytes))


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("kernel", [capi.KERNEL_AUTO, capi.KERNEL_BINNED])
def test_a_recorded_call_keeps_its_work_space(mode, kernel):
    """Larger calls after the recording get a work space of their own, also where they run while
    the graph replays."""
    print(f"streams: recorded call, mode {mode}, kernel {kernel}", flush=True)
    g, t = grid_tables(7)
    r = np.random.default_rng(7)
    dev = capi.Grid(t)
    Qs = [points(g, r, n) for n in (60_000, 20_000, 300_000, 900_000)]
    want = [[x.to_host() for x in device_call(dev, Q, capi.FP64, capi.KERNEL_TILE)[1:]] for Q in Qs]
    calls = [Call(dev, Q, capi.FP64) for Q in Qs]
    calls[0].run(None, kernel)  # leaves a work space and the tables
    graph = Graph(mode, lambda s: [calls[0].run(s, kernel), calls[1].run(s, kernel)])
    other = Stream()
    for big in (2, 3, 2):
        for c in calls:
            clobber(c)
        calls[big].run(other, capi.KERNEL_BINNED)
        graph.replay()
        calls[big].run(other, capi.KERNEL_BINNED)
        graph.replay()
        capi.check(capi.lib().brille_device_sync())
        for k in (0, 1, big):
            for a, b in zip(calls[k].out, want[k]):
                np.testing.assert_array_equal(a.to_host(), b, err_msg=f"call {k}")


@pytest.mark.parametrize("spec,kernel,entry", [
    (5, capi.KERNEL_TILE, "brille_ir_interpolate_at"), (5, capi.KERNEL_BINNED, "brille_ir_interpolate_at"),
    (3, capi.KERNEL_BINNED, "brille_ir_interpolate_at"), (3, capi.KERNEL_BINNED, "brille_ir_interpolate_at_noalloc")])
def test_a_recorded_call_keeps_its_tables_over_a_sort(spec, kernel, entry):
    """The graph goes on giving what its handle gave when it was recorded: unsorted, then sorted."""
    print(f"streams: recorded before a sort, grid {spec}, kernel {kernel}, {entry}", flush=True)
    g, t = grid_tables(spec, 300.0)
    t["values"], t["vectors"], _ = S.shuffled_modes(t, seed=4)
    dev = capi.Grid(t)
    Q = points(g, np.random.default_rng(8), 3_000)
    graphs = []
    for _ in range(2):
        want = [x.to_host() for x in device_call(dev, Q, capi.FP64, capi.KERNEL_BINNED)[1:]]
        call = Call(dev, Q, capi.FP64)
        graphs.append((Graph(1, lambda s: call.run(s, kernel, entry)), call, want))
        dev.sort()
        device_call(dev, Q, capi.FP64, capi.KERNEL_BINNED)  # its tables anew
        for graph, c, w in graphs * 2:
            clobber(c)
            graph.replay()
            capi.check(capi.lib().brille_device_sync())
            for a, b in zip(c.out, w):
                np.testing.assert_array_equal(a.to_host(), b)
    assert not np.array_equal(graphs[0][2][1], graphs[1][2][1])
