"""Grids with a PermutationTable on every payload layout: the specialised sums
and the row and factor tables follow the permutations exactly like the oracle
(PermutationTable::safe_get, src/permutation_table.hpp:193-198).  Needs an MI355X.
"""
import ctypes as C

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S
from oracle import oracle as O
from test_gpu_sort import device_table, oracle_table

pytestmark = pytest.mark.gpu


def small_tables(kind):
    """2, 4 atoms (one lane per mode), 12, 24 atoms (atom by atom), scalars of 2 and of 20 elements."""
    sp = dict(S.batch_specs(16)[{"a2": 3, "a4": 7, "a12": 2, "a24": 5}.get(kind, 3)], v_target=400.0)
    g = S.batch_grid(sp)
    t = S.batch_layout_tables(g, sp)
    if kind.startswith("s"):
        t.update(vectors_elements=[int(kind[1:]), 0, 0], vectors_rotates_like=0)
    t["values"], t["vectors"], order = S.shuffled_modes(t, seed=4)
    return t, order


def points(t, r, n):
    rlu = np.linalg.solve(np.asarray(t["outer_to_xyz"]).reshape(3, 3), np.asarray(t["vertices"]).T).T
    Q = r.uniform(-3, 3, size=(n, 3))
    k = r.integers(0, len(rlu), size=(n, 2))
    Q[::4] = 0.5 * (rlu[k[::4, 0]] + rlu[k[::4, 1]])  # irreducible already, some on cell faces
    Q[1::8] = rlu[k[1::8, 0]]
    return Q


def noalloc(dev, Q, precision):
    n = len(Q)
    vs, cs = dev.out_shapes(n)
    f32 = precision == capi.FP32
    dQ = capi.DeviceArray.from_host(Q)
    dv = capi.DeviceArray(vs, np.float32 if f32 else np.float64)
    dc = capi.DeviceArray(cs, np.complex64 if f32 else np.complex128)
    o = capi.RunOpts(0, precision, 0, capi.MEM_DEVICE, capi.KERNEL_BINNED, 1)
    capi.check(capi.lib().brille_ir_interpolate_at_noalloc(dev.h, dQ.ptr, n, C.byref(o), dv.ptr, dc.ptr, None, None))
    return dv.to_host(), dc.to_host()


@pytest.mark.parametrize("kind", ["a2", "a4", "a12", "a24", "s2", "s20"])
def test_sorted_payloads_match_the_oracle(kind):
    print(f"sorted layouts: {kind}", flush=True)
    t, _ = small_tables(kind)
    r = np.random.default_rng(17)
    Q = points(t, r, 3001)
    dev = capi.Grid(t)
    # tables built before the sort must not outlive it
    dev.ir_interpolate_at(Q[:100], precision=capi.FP64, kernel=capi.KERNEL_BINNED)
    dev.sort()
    perm = dev.permutations()
    assert len(perm[2]) > 1
    rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, nthreads=8, perm=perm)
    assert rc == 0
    got = {}
    for prec, tol in ((capi.FP64, 1e-12), (capi.FP32, 1e-5)):
        for name, f in (("noalloc", lambda: noalloc(dev, Q, prec)),
                        ("tile", lambda: dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)),
                        ("binned", lambda: dev.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_BINNED)),
                        ("tile with table", lambda: dev.ir_interpolate_at(Q, precision=prec,
                                                                          kernel=capi.KERNEL_TILE))):
            print(f"  {name} {prec}", flush=True)
            v, c = (x.reshape(o.shape) for x, o in zip(f(), (ov, oc)))
            assert np.max(np.abs(v - ov)) <= tol * np.abs(ov).max(), name
            assert np.max(np.abs(c - oc)) <= tol * np.abs(oc).max(), name
            if prec in got:
                np.testing.assert_array_equal(v, got[prec][0], err_msg=name)
                np.testing.assert_array_equal(c, got[prec][1], err_msg=name)
            got[prec] = (v, c)


@pytest.mark.parametrize("kind", ["a2", "a12", "s2"])
def test_random_permutations_of_a_few_pairs(kind):
    """Keys for some pairs only, and permutations unlike any assignment."""
    print(f"sorted layouts: random {kind}", flush=True)
    t, _ = small_tables(kind)
    V, B = len(t["vertices"]), int(t["branches"])
    r = np.random.default_rng(3)
    Q = points(t, r, 2000)
    rc, _, _, aux, _ = O.ir_interpolate_at(t, Q, nthreads=8)
    used = [aux["iw_index"][:, 0].astype(np.uint64) * V + aux["iw_index"][:, k] for k in range(1, 8)]
    keys = np.unique(np.concatenate(used))
    keys = np.sort(r.choice(keys, size=len(keys) // 2, replace=False))
    perms = np.array([r.permutation(B) for _ in range(9)], np.uint32)
    perm = (keys, r.integers(0, 9, size=len(keys)).astype(np.uint32), perms)
    rc, ov, oc, _, _ = O.ir_interpolate_at(t, Q, nthreads=8, perm=perm)
    assert rc == 0
    dev = capi.Grid(t, perm=perm)
    for kernel in (capi.KERNEL_PLAIN, capi.KERNEL_TILE, capi.KERNEL_BINNED):
        v, c = (x.reshape(o.shape) for x, o in zip(dev.ir_interpolate_at(Q, kernel=kernel), (ov, oc)))
        assert np.max(np.abs(v - ov)) <= 1e-12 * np.abs(ov).max(), kernel
        # a permuted pair's overlap can be small: its antiphase then carries the products' rounding
        assert np.max(np.abs(c - oc)) <= 1e-11 * np.abs(oc).max(), kernel


def test_a_batch_follows_a_member_sorted_after_its_first_run():
    print("sorted layouts: batch", flush=True)
    devs, Qs = [], []
    r = np.random.default_rng(9)
    for kind in ("a2", "a12", "s2"):
        t, _ = small_tables(kind)
        devs.append(capi.Grid(t))
        Qs.append(points(t, r, 700))
    off = np.concatenate([[0], np.cumsum([len(q) for q in Qs])]).astype(np.uint64)
    dQ = capi.DeviceArray.from_host(np.vstack(Qs))
    b = capi.Batch(devs)
    for prec in (capi.FP64, capi.FP32):
        vals, vecs = b.outputs(off, prec)
        capi.check(b.run(dQ, off, vals, vecs, precision=prec))
    for d in devs:
        d.sort()
    for prec in (capi.FP64, capi.FP32):
        vals, vecs = b.outputs(off, prec)
        capi.check(b.run(dQ, off, vals, vecs, precision=prec))
        for d, Q, v, c in zip(devs, Qs, vals, vecs):
            tv, tc = d.ir_interpolate_at(Q, precision=prec, kernel=capi.KERNEL_TILE)
            np.testing.assert_array_equal(v.to_host(), tv.reshape(v.shape))
            np.testing.assert_array_equal(c.to_host(), tc.reshape(c.shape))


@pytest.mark.parametrize("kind,spread", [("a2", 1e-10), ("a4", 1e-11), ("a2", 1e-6)])
def test_sort_of_near_ties_takes_the_exact_costs(kind, spread):
    """At some vertices two modes' vectors differ by `spread`: below the lead the one-kernel
    assignment asks for, such pairs go to the stored cost matrices and the solver; the table stays
    the oracle's.  No two such vertices share a cell: two near-equal modes on both sides swap at a
    cost of spread squared, a tie; and values that differ alone tie too, two absolute differences
    summed crosswise being the same sum."""
    print(f"sort near ties: {kind} {spread}", flush=True)
    t, _ = small_tables(kind)
    r = np.random.default_rng(12)
    vals, vecs = np.array(t["values"]), np.array(t["vectors"])
    B = vals.shape[1]
    near = O.sort_keys(t)
    near = np.stack([near // len(vals), near % len(vals)], 1).astype(np.int64)
    free = np.ones(len(vals), bool)
    for v in r.permutation(len(vals)):
        if not free[v]:
            continue
        free[near[near[:, 0] == v, 1]] = False
        a, b = r.choice(B, 2, replace=False)
        vals[v, b] = vals[v, a]
        vecs[v, b] = vecs[v, a] + spread * (r.normal(size=vecs.shape[2]) + 1j * r.normal(size=vecs.shape[2]))
    t["values"], t["vectors"] = vals, vecs
    keys, perms = oracle_table(t, nthreads=8)
    dev = capi.Grid(t)
    dev.sort()
    gk, gp = device_table(dev)
    np.testing.assert_array_equal(gk, keys)
    np.testing.assert_array_equal(gp, perms)


@pytest.mark.parametrize("value", [np.nan, np.inf, 1e200, 0.0])
def test_sort_of_values_beyond_the_cheap_costs(value):
    """A NaN or an overflowing vector reaches the literal costs, which report it; zero norms are sorted."""
    print(f"sort of {value}", flush=True)
    t, _ = small_tables("a2")
    t["vectors"] = np.array(t["vectors"])
    t["vectors"][7, 2] = value
    dev = capi.Grid(t)
    if value == 0.0:
        dev.sort()
        keys, perms = oracle_table(t, nthreads=8)
        gk, gp = device_table(dev)
        np.testing.assert_array_equal(gk, keys)
        np.testing.assert_array_equal(gp, perms)
    else:
        with pytest.raises(capi.BrilleError):
            dev.sort()
        # the grid stays usable without a table
        assert len(dev.permutations()[0]) == 0
