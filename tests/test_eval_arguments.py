"""Arguments that the flux and fit evaluations refuse before they reach the
device (no GPU needed)."""
import ctypes as C

import pytest

FS_E_ARG = -1


@pytest.fixture(scope="module")
def L():
    from fluidsim_amd import lib

    return lib.load()


def _call(L, name, n, a, out):
    if name == "fs_eval_fits":
        return L.fs_eval_fits(10.0, n, a, out)
    if name == "fs_eval_flux_noalloc":
        return L.fs_eval_flux_noalloc(n, a, out, 0)
    return getattr(L, name)(n, a, out)


@pytest.mark.parametrize("name", ["fs_eval_flux", "fs_eval_dfdph", "fs_eval_fits",
                                  "fs_eval_flux_noalloc"])
@pytest.mark.parametrize("n", [1, 16, 200])
def test_null_pointers_are_refused(L, name, n):
    buf = (C.c_double * (12 * n))()
    for a, out in ((None, buf), (buf, None), (None, None)):
        assert _call(L, name, n, a, out) == FS_E_ARG, (a is None, out is None)
        assert b"null" in L.fs_last_error()
    assert _call(L, name, 0, None, None) == 0
