"""Arguments that the flux and fit evaluations refuse before they reach the
device (no GPU needed)."""
import ctypes as C
import os
import shutil
import subprocess
import sys

import pytest

FS_E_ARG = -1
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


SHIM = r"""
/* the HIP calls of an evaluation on a device with id 64, one past the last that has
   a staging array; an allocation is reported */
#include <stddef.h>
#include <stdio.h>
int hipGetDevice(int* d) { *d = 64; return 0; }
int hipMalloc(void** p, size_t n) { (void)p; (void)n; puts("hipMalloc"); fflush(stdout); return 2; }
"""


def test_noalloc_does_not_allocate_on_a_device_without_the_array(tmp_path):
    if not shutil.which("gcc"):
        pytest.skip("gcc not available")
    (tmp_path / "shim.c").write_text(SHIM)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "shim.c")], check=True)
    code = ("import ctypes as C\nfrom fluidsim_amd import lib\nL = lib.load()\n"
            "a, o = (C.c_double * 1400)(), (C.c_double * 200)()\n"
            "print([f(n, a, o, *x) for n in (1, 200) for f, x in\n"
            "       ((L.fs_eval_flux_noalloc, (0,)), (L.fs_eval_flux, ()))])\n")
    before = os.environ.get("LD_PRELOAD", "")
    env = dict(os.environ, LD_PRELOAD=" ".join(filter(None, [so, before])))
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, check=True,
                         capture_output=True, text=True).stdout.split("\n")
    # (the other entry point takes its allocation there, and reports its failure)
    assert out[:3] == ["hipMalloc", "hipMalloc", "[-1, -6, -1, -6]"], out
