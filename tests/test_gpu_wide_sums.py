"""Node-ordered sums of wide Gamma rows, atom by atom: a point's records are
assembled in LDS and written as one run of 16-byte pieces (8-byte where a
record's start or length is no multiple of 16), in blocks of whole mode passes.

Shapes at the edges of a pass: one mode and a remainder, records of odd length,
passes cut short so that they end on a 64-byte granule, one mode per wave, more
modes than a block takes.  FP64 within 1e-12 of the oracle's scale, FP32 within
1e-5, and both bit for bit the fused kernel's.  Needs an MI355X.
"""
import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def payload(atoms, modes, one_to_one, seed):
    sp = dict(S.batch_specs(16)[3], v_target=2000.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    t = dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs)
    V, G = len(t["vertices"]), np.asarray(t["gamma_F0"]).shape[1]
    r = np.random.default_rng(seed)
    F0 = np.stack([r.permutation(atoms) for _ in range(G)], 1).astype(np.uint32)
    if not one_to_one:
        F0[1, G // 2:] = F0[0, G // 2:]
    t.update(values=r.normal(size=(V, modes, 1)), values_elements=[1, 0, 0], branches=modes,
             vectors=r.normal(size=(V, modes, 3 * atoms)) + 1j * r.normal(size=(V, modes, 3 * atoms)),
             vectors_elements=[0, 3 * atoms, 0], gamma_F0=F0,
             gamma_vector_index=r.integers(0, 7, size=(atoms, G)).astype(np.uint32),
             gamma_vectors=r.normal(size=(7, 3)))
    return t, F0


@pytest.mark.parametrize("atoms,modes", [(5, 13), (5, 12), (12, 9), (21, 7), (7, 90), (24, 1), (24, 41), (42, 3)])
def test_node_ordered_records_of_every_shape(atoms, modes):
    print(f"wide sums: {atoms} atoms, {modes} modes", flush=True)
    t, _ = payload(atoms, modes, True, 10 * atoms + modes)
    dev = capi.Grid(t)
    for n in (1, 65, 1500):
        Q = np.random.default_rng(n).uniform(-3, 3, size=(n, 3))
        rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, nthreads=8)
        assert rc == 0
        for prec, tol in ((capi.FP64, 1e-12), (capi.FP32, 1e-5)):
            bv, bc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_BINNED)
            tv, tc = dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
            np.testing.assert_array_equal(bv, tv)
            np.testing.assert_array_equal(bc, tc)
            assert np.max(np.abs(bv - ov)) <= tol * np.abs(ov).max(), (n, prec)
            assert np.max(np.abs(bc - oc)) <= tol * np.abs(oc).max(), (n, prec)


def test_operations_that_map_two_atoms_to_one():
    """No whole record to write: these payloads keep the sums that store atom by atom."""
    print("wide sums: two atoms to one", flush=True)
    t, F0 = payload(5, 7, False, 3)
    dev = capi.Grid(t)
    Q = np.random.default_rng(1).uniform(-3, 3, size=(700, 3))
    rc, _, oc, oaux, _ = O.ir_interpolate_at(t, Q, nthreads=8)
    assert rc == 0
    for kernel in (capi.KERNEL_BINNED, capi.KERNEL_TILE):
        _, c = dev.ir_interpolate_at(Q, precision=capi.FP64, kernel=kernel)
        c, o = c.reshape(700, 7, 5, 3), oc.reshape(700, 7, 5, 3)
        for p, op in enumerate(oaux["invrot"]):
            once = [a for a in range(5) if np.count_nonzero(F0[:, op] == a) == 1]
            assert np.max(np.abs(c[p][:, once] - o[p][:, once])) <= 1e-12 * np.abs(o).max()
