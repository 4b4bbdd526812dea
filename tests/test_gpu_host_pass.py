"""hp_bound_pass_host (host records in, a plan that lives for the call in one
allocation, records out) against hp_plan_run on device copies of the same
records: the kernels and the order of their sums are the same, so every field
is identical."""
import numpy as np
import pytest

import halopot
from halopot import catalog
from gpu_util import run_plan

pytestmark = pytest.mark.gpu


def _mixed():
    return catalog.small_batch(seed=81, n_halos=60, lo=2, hi=4000, potential_only=0.2)


def _large():
    """Calls above the sort's and the per-call kernels' bounds (16,384
    records), and over 32,768 records together."""
    return catalog.small_batch(seed=82, n_halos=3, lo=17_000, hi=25_000)


def _one():
    return catalog.small_batch(seed=83, n_halos=1, lo=134, hi=135, contam=0.0)


def _empty_calls():
    cat = catalog.small_batch(seed=84, n_halos=9, lo=5, hi=900)
    h = np.zeros(12, cat.halos.dtype)
    h[[1, 2, 3, 4, 6, 7, 8, 9, 10]] = cat.halos
    h["first"][[0, 5, 11]] = [0, cat.halos["first"][4], cat.n_records]
    cat.halos = h
    return cat


def _no_calls():
    cat = _one()
    cat.po, cat.halos = cat.po[:0].copy(), cat.halos[:0].copy()
    return cat


OPTIONS = {
    "default": {},
    "per_call": {"per_call": 1},
    "graph": {"use_graph": 1},
    "auto": {"method": halopot.METHOD_AUTO},
    "direct": {"method": halopot.METHOD_DIRECT},
    "f64": {"accumulate": halopot.ACC_F64},
}


@pytest.mark.parametrize("opts", OPTIONS)
@pytest.mark.parametrize("make", [_mixed, _large, _one, _empty_calls, _no_calls])
@pytest.mark.parametrize("want_bound", [True, False])
def test_host_pass_matches_plan_run(make, opts, want_bound):
    cat = make()
    cat.po["flags"] = np.arange(cat.n_records, dtype=np.int32)
    o = halopot.options(**OPTIONS[opts])
    po_d, h_d, bound_d, _ = run_plan(cat, o)
    po, h = cat.po.copy(), cat.halos.copy()
    bound = halopot.bound_pass_host(po, h, o, want_bound=want_bound)
    for f in po.dtype.names:
        np.testing.assert_array_equal(po[f], po_d[f], err_msg=f)
    for f in h.dtype.names:
        np.testing.assert_array_equal(h[f], h_d[f], err_msg=f)
    if want_bound:
        np.testing.assert_array_equal(bound, bound_d)
    else:
        assert bound is None


@pytest.mark.parametrize("extra", [-1, 1])
def test_host_pass_refuses_other_record_counts(extra):
    cat = _mixed()
    halopot.set_config(cat.params)
    po = np.zeros(cat.n_records + 1, cat.po.dtype)
    po[:-1] = cat.po
    po = po[:cat.n_records + extra].copy()
    before = po.tobytes()
    with pytest.raises(halopot.HalopotError, match="cover"):
        halopot.bound_pass_host(po, cat.halos.copy())
    assert po.tobytes() == before
