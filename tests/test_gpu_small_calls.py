"""Calls of few points: the fused kernel cuts its tiles by the call's size and
splits the modes of wide rows, and wide Gamma rows form their antiphases
atom by atom where no factor table holds them.

Every size must give the oracle's results (FP64 within 1e-12 relative, FP32
within 1e-5 of the scale), at the edges of the tiles and on points without a
table block (grid vertices and cell edges, where the first slot weighs
nothing).  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from conftest import CUBE, POLY, hand_trellis, tet_record
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 31, 33, 64, 65, 255, 257, 2049)


def points(g, r, n):
    """Uniform Q with every third point on a vertex or on the edge of two neighbouring vertices."""
    Q = r.uniform(-3, 3, size=(n, 3))
    rlu = np.asarray(g.rlu)
    k = r.integers(0, len(rlu) - 1, size=n)
    special = np.where(r.random((n, 1)) < 0.5, rlu[k], 0.5 * (rlu[k] + rlu[k + 1]))
    Q[::3] = special[::3]
    return Q


# atoms 2 and 4 (one lane per mode), 12 (5 modes a wave), 24 (2 modes a wave)
@pytest.mark.parametrize("spec", [3, 7, 2, 5])
def test_every_call_size_matches_the_oracle(spec):
    print(f"small calls: grid {spec}", flush=True)
    sp = dict(S.batch_specs(16)[spec], v_target=600.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    t = dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)
    dev = capi.Grid(t)
    r = np.random.default_rng(31 + spec)
    for n in SIZES:
        print(f"  n={n} B={sp['modes']}", flush=True)
        Q = points(g, r, n)
        rc, ov, oc, oaux, _ = O.ir_interpolate_at(t, Q, nthreads=8)
        assert rc == 0
        gv, gc, gaux = dev.ir_interpolate_at(Q, precision=capi.FP64, kernel=capi.KERNEL_TILE, aux=True)
        for k in ("tau", "rot", "invrot", "node", "tet", "n_iw", "iw_index", "iw_weight", "ir_q"):
            np.testing.assert_array_equal(gaux[k], oaux[k], err_msg=f"n={n} {k}")
        assert np.max(np.abs(gv - ov)) <= 1e-12 * np.abs(ov).max(), n
        assert np.max(np.abs(gc - oc)) <= 1e-12 * np.abs(oc).max(), n
        fv, fc = dev.ir_interpolate_at(Q, precision=capi.FP32, kernel=capi.KERNEL_TILE)
        assert np.max(np.abs(fv - ov)) <= 1e-5 * np.abs(ov).max(), n
        assert np.max(np.abs(fc - oc)) <= 1e-5 * np.abs(oc).max(), n
        for prec, (tv, tc) in ((capi.FP64, (gv, gc)), (capi.FP32, (fv, fc))):
            bv, bc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_BINNED)
            np.testing.assert_array_equal(bv, tv)
            np.testing.assert_array_equal(bc, tc)
            # the first binned call built the factor table: the fused kernel now reads it
            av, ac = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
            np.testing.assert_array_equal(av, tv)
            np.testing.assert_array_equal(ac, tc)


def test_a_failing_point_is_reported_once_by_every_split():
    """Modes split over several blocks of one tile: only the first reports, so the count stays exact."""
    print("small calls: errors", flush=True)
    sp = dict(S.batch_specs(16)[5], v_target=600.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    dev = capi.Grid(dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs))
    Q = np.random.default_rng(5).uniform(-3, 3, size=(5, 3))
    Q[3] = np.nan
    rc, v, c, aux = dev.run_device(Q, precision=capi.FP32, kernel=capi.KERNEL_TILE, check=False)
    assert rc == 0 and list(np.nonzero(aux["status"])[0]) == [3]
    assert np.all(v[3] == 0) and np.all(c[3] == 0) and np.all(np.isfinite(v))
    with pytest.raises(capi.BrilleError, match="Not all points inside Brillouin zone"):
        dev.ir_interpolate_at(Q, precision=capi.FP32, kernel=capi.KERNEL_TILE)


def test_wide_rows_of_neighbouring_cells_without_a_table():
    """A cube and the first tetrahedron of the node beside it, summed one after the other in node
    order on a handle that never built its factor table: each keeps its own rows."""
    print("small calls: neighbouring cells", flush=True)
    corner = [(1, 0, 0), (2, 0, 0), (1, 1, 0), (1, 0, 1)]
    t = hand_trellis({(0, 0, 0): CUBE, (1, 0, 0): POLY}, {(1, 0, 0): [corner]})
    V, A, B, G = len(t["vertices"]), 5, 3, len(np.asarray(t["inverse_index"]))
    r = np.random.default_rng(8)
    t.update(values=r.normal(size=(V, B, 1)), values_elements=[1, 0, 0], branches=B,
             vectors=r.normal(size=(V, B, 3 * A)) + 1j * r.normal(size=(V, B, 3 * A)), vectors_elements=[0, 3 * A, 0],
             vectors_rotates_like=2, vectors_length_unit=3,
             gamma_F0=np.repeat(np.arange(A, dtype=np.uint32)[:, None], G, 1),
             gamma_vector_index=np.zeros((A, G), np.uint32), gamma_vectors=np.zeros((1, 3)),
             gamma_cart_rotations=np.tile(np.eye(3).ravel(), (G, 1)))
    Q = np.vstack([r.uniform(0.1, 0.9, size=(40, 3)), [1.05, 0.05, 0.05] + r.uniform(0, 0.25, size=(40, 3))])
    rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, no_move=True)
    assert rc == 0
    dev = capi.Grid(t)
    n = len(Q)
    dQ, dv, dc = (capi.DeviceArray.from_host(Q), capi.DeviceArray((n, B, 1), np.float64),
                  capi.DeviceArray((n, B, 3 * A), np.complex128))
    o = capi.RunOpts(1, capi.FP64, 0, capi.MEM_DEVICE, capi.KERNEL_BINNED, 1)
    capi.check(capi.lib().brille_ir_interpolate_at_noalloc(dev.h, dQ.ptr, n, C.byref(o), dv.ptr, dc.ptr, None, None))
    assert np.max(np.abs(dv.to_host() - ov)) <= 1e-12 * np.abs(ov).max()
    assert np.max(np.abs(dc.to_host() - oc.reshape(n, B, -1))) <= 1e-12 * np.abs(oc).max()


@pytest.mark.parametrize("height", [0.3, 1e-2, 1e-4, 1e-7, 1e-11])
def test_flat_tetrahedra_are_located_like_the_oracle(height):
    """A tetrahedron split by a point `height` above its base: the FP32 forms that pass over the
    node's other tetrahedra must not pass over a flat one that holds the point."""
    print(f"small calls: flat tetrahedra {height}", flush=True)
    a, b, c, d, e = (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)
    t = hand_trellis({(0, 0, 0): POLY}, {(0, 0, 0): [(e, b, c, d), (a, b, c, e), (a, c, d, e), (a, d, b, e)]})
    # vertex e moves to `height` above the middle of face b, c, d
    apex = np.array([1.0, 1.0, 1.0]) * (1 / 3 - height)
    vid = int(np.nonzero((t["vertices"] == e).all(1))[0][0])
    t["vertices"] = np.array(t["vertices"])
    t["vertices"][vid] = apex
    rec = [tet_record(t["vertices"][v]) for v in t["tet_vertices"]]
    tv = np.array(t["tet_vertices"])
    for k, v in enumerate(tv):  # the moved apex can turn a tetrahedron over
        p = t["vertices"][v]
        if np.linalg.det(p[:3] - p[3]) < 0:
            tv[k] = v[[0, 1, 3, 2]]
    t["tet_vertices"] = tv
    t["tet_circumsphere"] = np.array([np.append(x[0][:3], x[0][3]) for x in rec])
    t["tet_volume"] = np.array([x[1] for x in rec])
    t["values"] = np.array(t["vertices"])[:, None, :].copy()
    r = np.random.default_rng(4)
    w = r.dirichlet(np.ones(4), size=600)
    Q = w @ np.array([a, b, c, d], float)
    w2 = r.dirichlet(np.ones(4), size=600)
    Q = np.vstack([Q, w2 @ np.array([apex, b, c, d], float)])  # inside the flat one
    rc, ov, _, oaux, _ = O.ir_interpolate_at(t, Q, no_move=True)
    assert rc == 0
    dev = capi.Grid(t)
    for kernel in (capi.KERNEL_TILE, capi.KERNEL_BINNED):
        gv, _, gaux = dev.ir_interpolate_at(Q, no_move=True, kernel=kernel, aux=dict(tau=False))
        for k in ("node", "tet", "n_iw", "iw_index", "iw_weight"):
            np.testing.assert_array_equal(gaux[k], oaux[k], err_msg=f"{kernel} {k}")
        np.testing.assert_allclose(gv, ov, atol=1e-12)


def device_call(dev, Q, precision, kernel, stream=None, out=None):
    n = len(Q)
    vs, cs = dev.out_shapes(n)
    f32 = precision == capi.FP32
    dQ = capi.DeviceArray.from_host(Q)
    dv, dc = out or (capi.DeviceArray(vs, np.float32 if f32 else np.float64),
                     capi.DeviceArray(cs, np.complex64 if f32 else np.complex128))
    o = capi.RunOpts(0, precision, 0, capi.MEM_DEVICE, kernel, 0 if stream else 1)
    capi.check(capi.lib().brille_ir_interpolate_at(dev.h, dQ.ptr, n, C.byref(o), dv.ptr, dc.ptr, None, stream))
    return dQ, dv, dc


@pytest.mark.parametrize("spec,precision,sizes", [
    (3, capi.FP32, (361_000, 361_200)), (3, capi.FP64, (194_000, 194_500)),
    (7, capi.FP32, (90_000, 90_300)), (7, capi.FP64, (48_500, 48_700)),
    (2, capi.FP32, (15_400, 15_500)), (5, capi.FP64, (770, 780)), (5, capi.FP32, (3_800, 3_900))])
def test_auto_agrees_with_the_fused_kernel_across_its_line(spec, precision, sizes):
    """The sizes on both sides of AUTO's choice between the fused kernel and the binned pipeline."""
    print(f"auto line: grid {spec} {precision}", flush=True)
    sp = dict(S.batch_specs(16)[spec], v_target=600.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    dev = capi.Grid(dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs))
    r = np.random.default_rng(2)
    for n in sizes:
        Q = points(g, r, n)
        tile = device_call(dev, Q, precision, capi.KERNEL_TILE)
        auto = device_call(dev, Q, precision, capi.KERNEL_AUTO)
        for a, b in zip(tile[1:], auto[1:]):
            np.testing.assert_array_equal(a.to_host(), b.to_host())


def test_an_auto_call_can_be_captured_first_and_after_a_binned_call():
    """Under capture nothing may be allocated: the first call of a handle stays with the fused
    kernel, one after an eager call of the same size takes the pipeline; both replay."""
    print("auto under capture", flush=True)
    lib = capi.lib()
    maps = open("/proc/self/maps").read().split()
    hip = C.CDLL(next(m for m in maps if "libamdhip64" in m))  # the runtime the library itself uses
    sp = dict(S.batch_specs(16)[7], v_target=600.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    t = dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)
    Q = points(g, np.random.default_rng(3), 120_000)
    want = device_call(capi.Grid(t), Q, capi.FP32, capi.KERNEL_TILE)
    for warm in (False, True):
        dev = capi.Grid(t)
        keep = device_call(dev, Q, capi.FP32, capi.KERNEL_AUTO if warm else capi.KERNEL_TILE)
        side, graph, replay = C.c_void_p(), C.c_void_p(), C.c_void_p()
        capi.check(lib.brille_stream_create(C.byref(side)))
        capi.check(lib.brille_device_sync())
        assert hip.hipStreamBeginCapture(side, 1) == 0  # thread-local mode
        o = capi.RunOpts(0, capi.FP32, 0, capi.MEM_DEVICE, capi.KERNEL_AUTO, 0)
        rc = lib.brille_ir_interpolate_at(dev.h, keep[0].ptr, len(Q), C.byref(o), keep[1].ptr, keep[2].ptr, None, side)
        assert hip.hipStreamEndCapture(side, C.byref(graph)) == 0
        capi.check(rc)
        assert hip.hipGraphInstantiate(C.byref(replay), graph, None, None, C.c_size_t(0)) == 0
        for _ in range(3):
            # eager work and clobbered outputs between the replays
            device_call(dev, Q[:500], capi.FP32, capi.KERNEL_TILE)
            for x in keep[1:]:
                junk = np.full(x.shape, 7, x.dtype)
                capi.check(lib.brille_memcpy_h2d(x.ptr, junk.ctypes.data_as(C.c_void_p), x.nbytes))
            assert hip.hipGraphLaunch(replay, side) == 0
            capi.check(lib.brille_stream_sync(side))
            for a, b in zip(want[1:], keep[1:]):
                np.testing.assert_array_equal(a.to_host(), b.to_host())
        assert hip.hipGraphExecDestroy(replay) == 0 and hip.hipGraphDestroy(graph) == 0
        capi.check(lib.brille_stream_destroy(side))
