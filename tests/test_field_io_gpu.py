"""Fields and evaluations across the C boundary (fs_set_field, fs_get_field,
fs_eval_flux, fs_eval_dfdph, fs_eval_fits): bitwise, at the sizes where the
transfer changes shape.  A plane is one piece up to 2^17 doubles, else pieces
of whole rows through two halves of the pinned block; an evaluation passes its
inputs in the launch's arguments (up to 112 doubles), through the fixed device
array (2 MiB in all), or through an allocation."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


# (nx + 2) (ny + 2): one odd-sized piece; exactly 2^17; two pieces; five with a
# short last one and odd rows; rows longer than half a piece
@pytest.mark.parametrize("nx,ny", [(9, 13), (510, 254), (361, 365), (701, 803), (1999, 70)])
def test_fields_cross_unchanged(nx, ny):
    from fluidsim_amd import Discharge, configs, lib

    L = lib.load()
    d = Discharge(configs.base(nx, ny))
    rng = np.random.default_rng(nx)
    P, R = nx + 2, ny + 2
    want = {f: rng.standard_normal((R, P)) for f in ("ni", "ne", "ph")}
    for f, a in want.items():  # consecutive writes reuse the pieces
        d.set(f, 1, a)
    for f, a in want.items():
        assert np.array_equal(d.get(f, 1), a), f
    wide = rng.standard_normal((R, P + 5))
    assert L.fs_set_field(d.h, lib.FIELDS["ne"], 1, _dp(wide), P + 5) == 0
    back = np.full((R, P + 3), -7.0)
    assert L.fs_get_field(d.h, lib.FIELDS["ne"], 1, _dp(back), P + 3) == 0
    assert np.array_equal(back[:, :P], wide[:, :P]) and np.all(back[:, P:] == -7.0)
    assert np.array_equal(d.get("ph", 1), want["ph"])
    d.close()


@pytest.mark.parametrize("name,ni,cuts", [("flux", 7, (1, 16, 17, 32768, 32769)),
                                          ("dfdph", 7, (1, 16, 17, 32768, 32769)),
                                          ("fits", 1, (1, 112, 113, 20164, 20165))])
def test_evaluations_do_not_depend_on_the_call_size(name, ni, cuts):
    from fluidsim_amd import discharge as D

    fn = {"flux": D.eval_flux, "dfdph": D.eval_dfdph, "fits": D.eval_fits}[name]
    rng = np.random.default_rng(5)
    n = cuts[-1]
    if ni == 7:
        a = 10.0 ** rng.uniform(-2, 2, (n, 7))
        a[:, 2] = rng.choice([-1.0, 1.0], n)
    else:
        a = 10.0 ** rng.uniform(-6, 2, n)
    full = fn(a)
    assert np.all(np.isfinite(full))
    for m in cuts[:-1]:
        assert np.array_equal(fn(a[:m]), full[:m]), m
