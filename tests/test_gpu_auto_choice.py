"""Which pipeline AUTO gives a call to, on both sides of its lines (read from the names of the
stages that a timed call reports), and the same results from either.  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from test_gpu_small_calls import device_call, points

pytestmark = pytest.mark.gpu


def scalar_grid(v_target, elements, values=1, modes=6):
    sp = dict(S.batch_specs(16)[3], v_target=float(v_target))
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    V = len(t["vertices"])
    r = np.random.default_rng(elements)
    t.update(values=r.normal(size=(V, modes, values)), values_elements=[values, 0, 0], branches=modes,
             vectors=r.normal(size=(V, modes, elements)) + 1j * r.normal(size=(V, modes, elements)),
             vectors_elements=[elements, 0, 0], vectors_rotates_like=0)
    return g, t


def takes_pipeline(dev, Q, precision, kernel=capi.KERNEL_AUTO):
    vs, cs = dev.out_shapes(len(Q))
    f32 = precision == capi.FP32
    dQ = capi.DeviceArray.from_host(Q)
    dv = capi.DeviceArray(vs, np.float32 if f32 else np.float64)
    dc = capi.DeviceArray(cs, np.complex64 if f32 else np.complex128)
    o, t = capi.RunOpts(0, precision, 0, capi.MEM_DEVICE, kernel, 1), capi.KernelTimes()
    capi.check(capi.lib().brille_time_ir_interpolate_at(dev.h, dQ.ptr, len(Q), C.byref(o), dv.ptr, dc.ptr, 1, None,
                                                        C.byref(t)))
    return t.names[0].value.startswith(b"k_bin")


# payloads above 8 MB; rows that the general sums read twice take the pipeline like any other,
# rows of one to four elements from the sizes where it pays
@pytest.mark.parametrize("elements,values,precision,n,binned", [
    (8, 1, capi.FP64, 270_000, True), (8, 1, capi.FP32, 270_000, True), (5, 1, capi.FP64, 270_000, True),
    (2, 2, capi.FP32, 270_000, True), (1, 1, capi.FP64, 2_200_000, False), (1, 1, capi.FP64, 2_400_000, True),
    (4, 1, capi.FP64, 270_000, False), (4, 1, capi.FP64, 300_000, True), (4, 1, capi.FP32, 1_050_000, False),
    (4, 1, capi.FP32, 1_100_000, True)])
def test_scalar_rows(elements, values, precision, n, binned):
    print(f"auto choice: {elements} elements, {values} values, {precision}, {n} points", flush=True)
    g, t = scalar_grid(250_000 if elements == 1 else 110_000, elements, values)
    row = 16 * 2 ** int(np.ceil(np.log2((2 * elements + values) / 4)))  # bytes of an FP32 payload row
    assert len(t["vertices"]) * 6 * row > 8 << 20
    dev = capi.Grid(t)
    Q = points(g, np.random.default_rng(3), n)
    assert takes_pipeline(dev, Q, precision) == binned
    auto = device_call(dev, Q, precision, capi.KERNEL_AUTO)
    tile = device_call(dev, Q, precision, capi.KERNEL_TILE)
    for a, b in zip(auto[1:], tile[1:]):
        np.testing.assert_array_equal(a.to_host(), b.to_host())


# grid, precision, points of a call above the line of work, points a cell that pay for the table
@pytest.mark.parametrize("spec,v_target,precision,n,per_cell", [
    (7, 30_000, capi.FP64, 60_000, 14), (7, 30_000, capi.FP32, 110_000, 24), (5, 1_000, capi.FP64, 1_000, 1.5),
    (5, 12_000, capi.FP32, 4_500, 2.5)])
def test_ordinary_calls_until_they_have_paid_for_the_table(spec, v_target, precision, n, per_cell):
    print(f"auto choice: table of grid {spec}, {precision}, {n} points", flush=True)
    sp = dict(S.batch_specs(16)[spec], v_target=float(v_target))
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    t = dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)
    cells = len(t["cube_vertices"]) + len(t["tet_vertices"]) // 2
    due = int(np.ceil(per_cell * cells / n))  # the call that builds it
    assert 1 < due < 60
    dev = capi.Grid(t)
    Q = points(g, np.random.default_rng(4), n)
    want = [x.to_host() for x in device_call(dev, Q, precision, capi.KERNEL_TILE)[1:]]
    for k in range(1, due + 2):
        assert takes_pipeline(dev, Q, precision) == (k >= due), k
        if k in (1, due):
            for a, b in zip(device_call(dev, Q[:n // 9], precision, capi.KERNEL_AUTO)[1:], want):
                np.testing.assert_array_equal(a.to_host(), b[:n // 9])
    for a, b in zip(device_call(dev, Q, precision, capi.KERNEL_AUTO)[1:], want):
        np.testing.assert_array_equal(a.to_host(), b)
    dev.fill(t)  # a new payload counts anew
    assert not takes_pipeline(dev, Q, precision)
    device_call(dev, Q, precision, capi.KERNEL_BINNED)  # a call that asks for the table
    assert takes_pipeline(dev, Q, precision)
