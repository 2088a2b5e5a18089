"""Edges of the calls: outputs that are only 8-byte aligned, host calls of more than one chunk of
2^20 points, and batch members whose operations map two atoms to one.  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from test_gpu_small_calls import device_call
from test_gpu_wide_sums import payload

pytestmark = pytest.mark.gpu


def tables(kind):
    """2 and 4 atoms, 5 and 12 atoms (atom by atom), scalars of 1, 2, 5 and 20 elements."""
    if kind in ("a5", "a12"):
        return payload(int(kind[1:]), 7, True, 5)[0]
    sp = dict(S.batch_specs(16)[{"a2": 3, "a4": 7}.get(kind, 3)], v_target=400.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    t = dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)
    if kind.startswith("s"):
        k, r = int(kind[1:]), np.random.default_rng(1)
        V, B = vals.shape[:2]
        t.update(vectors=r.normal(size=(V, B, k)) + 1j * r.normal(size=(V, B, k)), vectors_elements=[k, 0, 0],
                 vectors_rotates_like=0)
    return t


@pytest.mark.parametrize("kind", ["a2", "a4", "a5", "a12", "s1", "s2", "s5", "s20"])
@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32])
def test_outputs_aligned_to_eight_bytes(kind, precision):
    print(f"call edges: {kind} {precision}, outputs 8 bytes off", flush=True)
    dev = capi.Grid(tables(kind))
    n = 3001
    Q = np.random.default_rng(2).uniform(-3, 3, size=(n, 3))
    dQ = capi.DeviceArray.from_host(Q)
    f32 = precision == capi.FP32
    vs, cs = dev.out_shapes(n)
    vs, cs = (n, int(np.prod(vs[1:]))), (n, int(np.prod(cs[1:])))
    for kernel in (capi.KERNEL_TILE, capi.KERNEL_BINNED):
        want = device_call(dev, Q, precision, kernel)
        # rows before and after catch stores beyond the arrays
        bv = capi.DeviceArray.from_host(np.full((n + 4) * vs[1], 7, np.float32 if f32 else np.float64))
        bc = capi.DeviceArray.from_host(np.full((n + 4) * 2 * cs[1], 7, np.float32 if f32 else np.float64))
        o = capi.RunOpts(0, precision, 0, capi.MEM_DEVICE, kernel, 1)
        capi.check(capi.lib().brille_ir_interpolate_at(dev.h, dQ.ptr, n, C.byref(o), C.c_void_p(bv.ptr.value + 8),
                                                       C.c_void_p(bc.ptr.value + 8), None, None))
        for got, w, per in ((bv, want[1], 8 // (4 if f32 else 8)), (bc, want[2], 8 // (4 if f32 else 8))):
            flat, ref = got.to_host(), w.to_host().reshape(-1).view(got.dtype)
            np.testing.assert_array_equal(flat[per:per + ref.size], ref)
            assert (flat[:per] == 7).all() and (flat[per + ref.size:] == 7).all()


AUX = ("ir_q", "rot", "invrot", "node", "tet", "n_iw", "iw_index", "iw_weight", "status")


@pytest.mark.parametrize("kind", ["s1", "s5"])
def test_host_call_of_two_chunks(kind):
    print(f"call edges: {kind}, two chunks of host memory", flush=True)
    t = tables(kind)
    t.update(values=np.array(t["values"])[:, :2], vectors=np.array(t["vectors"])[:, :2], branches=2)
    dev = capi.Grid(t)
    n = (1 << 20) + 4099
    Q = np.random.default_rng(3).uniform(-3, 3, size=(n, 3))
    rc, dv, dc, daux = dev.run_device(Q, precision=capi.FP32, aux=AUX)
    assert rc == 0
    v, c, aux = dev.ir_interpolate_at(Q, precision=capi.FP32, aux=True)
    np.testing.assert_array_equal(v, dv)
    np.testing.assert_array_equal(c, dc)
    for k in AUX:
        np.testing.assert_array_equal(aux[k], daux[k], err_msg=k)
    Q[(1 << 20) + 77] = (1.5, np.nan, 0.25)
    with pytest.raises(capi.BrilleError, match=r"Not all points inside Brillouin zone.*\[1.5, -?nan, 0.25\]"):
        dev.ir_interpolate_at(Q, precision=capi.FP32)


def test_batch_members_whose_operations_map_two_atoms_to_one():
    print("call edges: batch of tables that are not one to one", flush=True)
    members = [payload(A, B, A == 12, 4) for A, B in ((5, 7), (12, 9), (2, 6))]
    devs = [capi.Grid(t) for t, _ in members]
    r = np.random.default_rng(6)
    Qs = [r.uniform(-3, 3, size=(n, 3)) for n in (900, 700, 800)]
    off = np.concatenate([[0], np.cumsum([len(q) for q in Qs])]).astype(np.uint64)
    dQ = capi.DeviceArray.from_host(np.vstack(Qs))
    b = capi.Batch(devs)
    for binned_min in (None, 1):
        b.set_schedule(tile_points=128, binned_min=binned_min)
        for prec in (capi.FP64, capi.FP32):
            vals, vecs = b.outputs(off, prec)
            capi.check(b.run(dQ, off, vals, vecs, precision=prec))
            for d, Q, v, c, (t, F0) in zip(devs, Qs, vals, vecs, members):
                rc, tv, tc, aux = d.run_device(Q, precision=prec, kernel=capi.KERNEL_TILE, aux=("invrot",))
                assert rc == 0
                np.testing.assert_array_equal(v.to_host(), tv)
                A = F0.shape[0]
                got, ref = (x.reshape(len(Q), -1, A, 3) for x in (c.to_host(), tc))
                for p, op in enumerate(aux["invrot"]):
                    once = [a for a in range(A) if np.count_nonzero(F0[:, op] == a) == 1]
                    np.testing.assert_array_equal(got[p][:, once], ref[p][:, once])


@pytest.mark.parametrize("atoms,modes", [(5, 13), (12, 9), (24, 41), (42, 3)])
def test_wide_tables_that_are_not_one_to_one(atoms, modes):
    """Element for element the fused kernel's results in every pipeline, and the elements no atom is
    mapped to are left as they were."""
    print(f"call edges: {atoms} atoms, {modes} modes, not one to one", flush=True)
    t, F0 = payload(atoms, modes, False, 10 * atoms + modes)
    dev = capi.Grid(t)
    for n in (1, 700):
        Q = np.random.default_rng(n).uniform(-3, 3, size=(n, 3))
        dQ = capi.DeviceArray.from_host(Q)
        for prec in (capi.FP64, capi.FP32):
            got = []
            for kernel in (capi.KERNEL_TILE, capi.KERNEL_BINNED, capi.KERNEL_TILE):  # without and with the table
                dv = capi.DeviceArray((n, modes), np.float32 if prec == capi.FP32 else np.float64)
                dc = capi.DeviceArray.from_host(np.full((n, modes, atoms, 3), 7, np.complex64 if prec == capi.FP32 else np.complex128))
                o = capi.RunOpts(0, prec, 0, capi.MEM_DEVICE, kernel, 1)
                capi.check(capi.lib().brille_ir_interpolate_at(dev.h, dQ.ptr, n, C.byref(o), dv.ptr, dc.ptr, None, None))
                got.append((dv.to_host(), dc.to_host()))
            rc, _, _, aux = dev.run_device(Q, precision=prec, aux=("invrot",))
            assert rc == 0
            for v, c in got[1:]:
                np.testing.assert_array_equal(v, got[0][0])
                for p, op in enumerate(aux["invrot"]):
                    count = np.bincount(F0[:, op], minlength=atoms)
                    np.testing.assert_array_equal(c[p][:, count == 1], got[0][1][p][:, count == 1])
                    assert (c[p][:, count == 0] == 7).all()
