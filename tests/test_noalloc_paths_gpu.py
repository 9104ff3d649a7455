"""GPU: fs_eval_flux_noalloc against a path that shares nothing with it but the
formula: slices of one call of fs_eval_flux / fs_eval_dfdph above 32768 entries,
which stages its inputs in an allocation.  (At up to 32768 entries these entry
points run the same code on the same fixed array.)  Sizes on both sides of the 16
entries that travel in the launch's arguments, and the largest."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


@pytest.mark.parametrize("dfdph", [0, 1])
def test_noalloc_equals_a_call_that_allocates(dfdph):
    from fluidsim_amd import lib

    L = lib.load()
    rng = np.random.default_rng(3 + dfdph)
    n = 32769
    a = np.ascontiguousarray(np.stack(
        [rng.standard_normal(n) * 10.0 ** rng.uniform(-14, 5, n), rng.uniform(0.2, 3.0, n),
         rng.choice([-1.0, 1.0], n), 10.0 ** rng.uniform(-3, 3, n), 10.0 ** rng.uniform(-2, 4, n),
         10.0 ** rng.uniform(-4, 8, n), 10.0 ** rng.uniform(-4, 8, n)], 1))
    full = np.full(n, -7.0)
    assert (L.fs_eval_dfdph if dfdph else L.fs_eval_flux)(n, _dp(a), _dp(full)) == 0
    for at, m in ((0, 32768), (5, 1537), (100, 17), (200, 16), (300, 1)):
        part, got = np.ascontiguousarray(a[at:at + m]), np.full(m, -7.0)
        assert L.fs_eval_flux_noalloc(m, _dp(part), _dp(got), dfdph) == 0
        # bits, infinities and NaN included
        assert np.array_equal(got.view(np.uint64), full[at:at + m].view(np.uint64)), m
