"""Host-memory calls: small ones have the kernels write to pinned memory, larger
ones send their results through a ring of pinned slots by several threads.
Bit for bit the device-memory call's results, for results of one byte range
up to more chunks than the ring has slots, and from several threads on one
handle.  Needs an MI355X.
"""
import threading

import numpy as np
import pytest

from brille_amd import capi
from brille_amd import synthetic as S

pytestmark = pytest.mark.gpu
AUX = ("ir_q", "rot", "invrot", "node", "tet", "n_iw", "iw_index", "iw_weight", "status")


def grid(spec=3):
    sp = dict(S.batch_specs(16)[spec], v_target=600.0)
    g = S.batch_grid(sp)
    vals, vecs = S.batch_payload(g, sp)
    return capi.Grid(dict(S.batch_layout_tables(g, sp), values=vals, vectors=vecs))


# one point; either side of 4 MB; the ring with one thread, with several and
# with more chunks than slots (600 bytes a point FP64 for grid 3, 83 000 for grid 5)
@pytest.mark.parametrize("spec,n", [(3, 1), (3, 5003), (3, 9001), (3, 45007), (5, 41), (5, 1501)])
def test_host_results_equal_device_results(spec, n):
    print(f"host calls: grid {spec}, {n} points", flush=True)
    dev = grid(spec)
    Q = np.random.default_rng(n).uniform(-3, 3, size=(n, 3))
    for prec in (capi.FP64, capi.FP32):
        rc, dv, dc, daux = dev.run_device(Q, precision=prec, aux=AUX)
        assert rc == 0
        for aux in (False, True):
            got = dev.ir_interpolate_at(Q, precision=prec, aux=aux)
            np.testing.assert_array_equal(got[0], dv)
            np.testing.assert_array_equal(got[1], dc)
        for k in AUX:
            np.testing.assert_array_equal(got[2][k], daux[k], err_msg=k)


def test_small_and_large_calls_from_threads_of_one_handle():
    print("host calls: threads", flush=True)
    dev = grid()
    sizes = (1, 300, 9001, 45007)
    Qs = [np.random.default_rng(k).uniform(-3, 3, size=(n, 3)) for k, n in enumerate(sizes)]
    want = [dev.run_device(Q)[1:3] for Q in Qs]
    bad = []

    def call(k):
        for _ in range(3):
            v, c = dev.ir_interpolate_at(Qs[k])
            if not (np.array_equal(v, want[k][0]) and np.array_equal(c, want[k][1])):
                bad.append(k)

    ts = [threading.Thread(target=call, args=(k,)) for k in range(len(sizes))]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad


@pytest.mark.parametrize("n", [3, 9001])
def test_errors_are_those_of_their_own_call(n):
    print(f"host calls: errors, {n} points", flush=True)
    dev = grid()
    Q = np.random.default_rng(n).uniform(-3, 3, size=(n, 3))
    bad = Q.copy()
    bad[n // 2] = np.nan
    with pytest.raises(capi.BrilleError, match="Not all points inside Brillouin zone"):
        dev.ir_interpolate_at(bad)
    v, c = dev.ir_interpolate_at(Q)
    assert np.isfinite(v).all() and np.isfinite(c).all()
