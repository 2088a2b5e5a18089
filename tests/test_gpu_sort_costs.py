"""Sorts whose costs leave the range of the one-kernel assignment: they take the literal costs, so
that the table stays the oracle's and what the reference's sum refuses is refused.  Needs an MI355X.
"""
import numpy as np
import pytest

from brille_amd import capi
from test_gpu_sort import device_table, oracle_table
from test_gpu_sorted_layouts import small_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1.0, 1.17e77, 1e-75])
def test_sort_of_vectors_whose_norms_product_overflows(scale):
    """Unit vectors times 1.17e77: |a|^2 |b|^2 is infinite, |a.b|^2 is not."""
    print(f"sort of vectors of length {scale}", flush=True)
    t, _ = small_tables("a2")
    r = np.random.default_rng(21)
    shape = np.asarray(t["vectors"]).shape
    u = r.normal(size=shape) + 1j * r.normal(size=shape)
    t["vectors"] = u / np.sqrt((np.abs(u) ** 2).sum(-1, keepdims=True)) * scale
    t["values"] = 0.3 * r.normal(size=np.asarray(t["values"]).shape)
    keys, perms = oracle_table(t, nthreads=8)
    dev = capi.Grid(t)
    dev.sort()
    gk, gp = device_table(dev)
    np.testing.assert_array_equal(gk, keys)
    np.testing.assert_array_equal(gp, perms)


@pytest.mark.parametrize("which,at", [("values", 1), ("values", 2), ("vectors", 0), ("vectors", 2)])
def test_sort_refuses_weights_that_are_not_finite(which, at):
    """An infinite weight of an absent term makes every cost a NaN, as in the reference's sum."""
    print(f"sort with an infinite weight: {which} {at}", flush=True)
    t, _ = small_tables("a2")
    dev = capi.Grid(t)
    w = [1.0, 1.0, 1.0]
    w[at] = np.inf
    with pytest.raises(capi.BrilleError):
        dev.sort(**{which + "_cost": capi.cost_info(weights=w)})
