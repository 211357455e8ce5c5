"""The molecule of each quartet of a batch class (csrc/batch_find.h, run on the
host): right for molecules without a quartet of the class in any place, and
found in no more reads than a search over the batch."""
import ctypes
import os

import numpy as np
import pytest

HC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hostcheck", "libhostcheck.so")


def _counts(kind):
    rng = np.random.default_rng(7)
    if kind == "one":
        return np.array([5])
    if kind == "none":
        return np.zeros(9, int)
    if kind == "marks":       # ends at, before and after multiples of 64
        return np.array([64, 63, 1, 65, 0, 127, 1, 0, 64, 0])
    if kind == "singles":     # many molecules to one wavefront
        return np.ones(1000, int)
    if kind == "runs":        # long runs without a quartet, also first and last
        c = np.zeros(5000, int)
        c[rng.choice(np.arange(40, 4900), 12, replace=False)] = rng.integers(1, 150, 12)
        return c
    return rng.integers(0, 90, 700) * (rng.random(700) < 0.5)


@pytest.mark.parametrize("kind", ["one", "none", "marks", "singles", "runs", "random"])
def test_quartet_molecules(kind):
    if not os.path.exists(HC):
        pytest.skip("host check harness not built (run __graft_entry__.build())")
    c = np.ascontiguousarray(_counts(kind), dtype=np.int64)
    want = np.repeat(np.arange(len(c)), c)
    got = np.full(max(len(want), 1), -1, dtype=np.int32)
    reads = ctypes.CDLL(HC).hc_quartet_molecules(len(c), c.ctypes.data_as(ctypes.POINTER(ctypes.c_longlong)),
                                                 got.ctypes.data_as(ctypes.POINTER(ctypes.c_int)))
    assert np.array_equal(got[:len(want)], want)
    assert reads <= int(np.ceil(np.log2(len(c) + 1)))
    if kind == "one":
        assert reads == 0
