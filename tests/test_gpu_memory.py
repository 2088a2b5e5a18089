"""A call that AUTO gives to the binned pipeline while the device has no memory left for the
pipeline's table: the fused kernel, which needs none, serves it.  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from test_gpu_small_calls import device_call, points
from test_gpu_streams import Call, clobber, hip_runtime

pytestmark = pytest.mark.gpu
LEAVE = 600 << 20  # bytes left free: enough for the runtime, less than the table


def free_bytes(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def take_memory(hip):
    """Allocations of the library's that leave about LEAVE bytes."""
    held, piece = [], 64 << 30
    while piece >= 64 << 20:
        p = C.c_void_p()
        if free_bytes(hip) < LEAVE + piece or capi.lib().brille_device_alloc(piece, C.byref(p)) != 0:
            piece //= 2
        else:
            held.append(p)
    return held


def test_auto_without_memory_for_the_table():
    print("auto without memory", flush=True)
    sp = dict(S.batch_specs(16)[7], v_target=120_000.0)
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    V, B, sc = len(t["vertices"]), int(t["branches"]), int(sum(t["vectors_elements"]))
    r = np.random.default_rng(1)
    t.update(values=r.normal(size=(V, B, 1)), vectors=r.normal(size=(V, B, sc)) + 1j * r.normal(size=(V, B, sc)))
    cells = len(t["cube_vertices"]) * 8 + len(t["tet_vertices"]) * 4
    assert cells * B * (2 * sc + 1) * 8 > LEAVE + (200 << 20)
    dev = capi.Grid(t)
    Q = points(g, r, 300_000)
    want = [x.to_host() for x in device_call(dev, Q, capi.FP64, capi.KERNEL_TILE)[1:]]
    call = Call(dev, Q, capi.FP64)
    hip = hip_runtime()
    held = take_memory(hip)
    print(f"  {free_bytes(hip) >> 20} MB left", flush=True)
    try:
        with pytest.raises(capi.BrilleError) as e:
            call.run(None, capi.KERNEL_BINNED)
        assert e.value.status == "DEVICE"
        clobber(call)
        call.run(None, capi.KERNEL_AUTO)
        capi.check(capi.lib().brille_device_sync())
    finally:
        for p in held:
            capi.lib().brille_device_free(p)
    for a, b in zip(call.out, want):
        np.testing.assert_array_equal(a.to_host(), b)
    clobber(call)
    call.run(None, capi.KERNEL_BINNED)  # the memory is there again
    capi.check(capi.lib().brille_device_sync())
    for a, b in zip(call.out, want):
        np.testing.assert_array_equal(a.to_host(), b)


def test_a_large_sort_gives_its_work_space_back():
    print("memory after a sort", flush=True)
    sp = dict(S.batch_specs(16)[7], v_target=120_000.0)
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    V, B, sc = len(t["vertices"]), 60, int(sum(t["vectors_elements"]))
    r = np.random.default_rng(2)
    values = np.tile(2.0 * np.arange(B)[:, None], (V, 1, 1))  # far apart: every pair keeps its order
    vectors = np.broadcast_to(r.normal(size=(1, B, sc)) + 1j * r.normal(size=(1, B, sc)), (V, B, sc))
    t.update(values=values, vectors=vectors, branches=B)
    dev = capi.Grid(t)
    hip = hip_runtime()
    before = free_bytes(hip)
    dev.sort()
    left = before - free_bytes(hip)
    keys, index, perms = dev.permutations()
    assert len(perms) == 1 and len(keys) > 1_500_000
    work = len(keys) // 2 * (36 + 2 * B)
    print(f"  {len(keys)} keys, work space {work >> 20} MB, {left >> 20} MB left with the handle", flush=True)
    # what stays: keys, their indices, the first key of every vertex, a word per cell slot
    cells = 8 * len(t["cube_vertices"]) + 4 * len(t["tet_vertices"])
    assert work > 128 << 20
    assert left <= 12 * len(keys) + 4 * (V + cells) + (16 << 20)
