"""Scalar rows of one to four elements with a PermutationTable in the binned sums:
every point the row table serves is summed from it, also where a row is a single
16-byte chunk (one element FP32), so that no point follows a slot permutation
that was never looked up.  Needs an MI355X.
"""
import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# modes: one, the usual, more than the block has lanes
@pytest.mark.parametrize("elements", [1, 2, 3, 4])
@pytest.mark.parametrize("modes", [1, 6, 300])
def test_permuted_scalar_rows_in_the_binned_sums(elements, modes):
    print(f"sorted rows: {elements} elements, {modes} modes", flush=True)
    sp = dict(S.batch_specs(16)[3], v_target=400.0)
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    V = len(t["vertices"])
    r = np.random.default_rng(10 * modes + elements)
    t.update(values=r.normal(size=(V, modes, 1)), values_elements=[1, 0, 0], branches=modes,
             vectors=r.normal(size=(V, modes, elements)) + 1j * r.normal(size=(V, modes, elements)),
             vectors_elements=[elements, 0, 0], vectors_rotates_like=0)
    Q = r.uniform(-3, 3, size=(1500, 3))
    rc, _, _, aux, _ = O.ir_interpolate_at(t, Q, nthreads=8)
    assert rc == 0
    used = [aux["iw_index"][:, 0].astype(np.uint64) * V + aux["iw_index"][:, k] for k in range(1, 8)]
    keys = np.unique(np.concatenate(used))
    perms = np.array([r.permutation(modes) for _ in range(9)], np.uint32)
    perm = (keys, r.integers(0, 9, size=len(keys)).astype(np.uint32), perms)
    rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, nthreads=8, perm=perm)
    assert rc == 0
    dev = capi.Grid(t, perm=perm)
    for prec, tol in ((capi.FP64, 1e-12), (capi.FP32, 1e-5)):
        bv, bc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_BINNED)
        tv, tc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
        np.testing.assert_array_equal(bv, tv)
        np.testing.assert_array_equal(bc, tc)
        assert np.max(np.abs(bv - ov)) <= tol * np.abs(ov).max()
        if elements == 1:  # one element's antiphase turns it onto the pivot: no cancelling overlap
            assert np.max(np.abs(bc - oc)) <= tol * np.abs(oc).max()


def sorted_grid(elements, values, atoms):
    sp = dict(S.batch_specs(16)[3], v_target=400.0)
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    V, G = len(t["vertices"]), np.asarray(t["gamma_F0"]).shape[1]
    r = np.random.default_rng(elements)
    modes, A = 7, elements // 3
    t.update(values=r.normal(size=(V, modes, values)), values_elements=[values, 0, 0], branches=modes,
             vectors=r.normal(size=(V, modes, elements)) + 1j * r.normal(size=(V, modes, elements)))
    if atoms:
        t.update(vectors_elements=[0, elements, 0], gamma_F0=np.stack([r.permutation(A) for _ in range(G)], 1).astype(np.uint32),
                 gamma_vector_index=r.integers(0, 7, size=(A, G)).astype(np.uint32), gamma_vectors=r.normal(size=(7, 3)))
    else:
        t.update(vectors_elements=[elements, 0, 0], vectors_rotates_like=0)
    dev = capi.Grid(t)
    dev.sort()
    perm = dev.permutations()
    return dev, t, perm, r


# either side of the longest sorted row a lane sums, and rows of more values than atoms
@pytest.mark.parametrize("elements,values,atoms", [(13, 1, False), (24, 1, False), (25, 1, False), (15, 6, True), (24, 9, True), (27, 10, True)])
def test_sorted_rows_around_the_longest_a_lane_sums(elements, values, atoms):
    print(f"sorted rows: {elements} elements, {values} values, atoms {atoms}", flush=True)
    dev, t, perm, r = sorted_grid(elements, values, atoms)
    for n in (1, 300, 20_000):
        Q = r.uniform(-3, 3, size=(n, 3))
        rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, nthreads=8, perm=perm)
        assert rc == 0
        for prec, tol in ((capi.FP64, 1e-12), (capi.FP32, 1e-5)):
            bv, bc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_BINNED)
            tv, tc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
            np.testing.assert_array_equal(bv, tv)
            np.testing.assert_array_equal(bc, tc)
            assert np.max(np.abs(bv - ov)) <= tol * np.abs(ov).max(), (n, prec)
            # an assigned pair's overlap can still be small, and the antiphase then carries the products' rounding
            assert np.max(np.abs(bc - oc)) <= 10 * tol * np.abs(oc).max(), (n, prec)


def test_a_batch_of_sorted_rows_around_the_longest_a_lane_sums():
    print("sorted rows: batch", flush=True)
    devs = [sorted_grid(*form)[0] for form in ((13, 1, False), (24, 1, False), (25, 1, False), (15, 6, True))]
    Qs = [np.random.default_rng(k).uniform(-3, 3, size=(600 + 100 * k, 3)) for k in range(len(devs))]
    off = np.concatenate([[0], np.cumsum([len(q) for q in Qs])]).astype(np.uint64)
    dQ = capi.DeviceArray.from_host(np.vstack(Qs))
    b = capi.Batch(devs)
    for binned_min in (None, 1):
        b.set_schedule(tile_points=128, binned_min=binned_min)
        for prec in (capi.FP64, capi.FP32):
            vals, vecs = b.outputs(off, prec)
            capi.check(b.run(dQ, off, vals, vecs, precision=prec))
            for d, Q, v, c in zip(devs, Qs, vals, vecs):
                tv, tc = d.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
                np.testing.assert_array_equal(v.to_host(), tv.reshape(v.shape))
                np.testing.assert_array_equal(c.to_host(), tc.reshape(c.shape))
