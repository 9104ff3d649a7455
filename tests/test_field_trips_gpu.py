"""GPU: fields cross the boundary by a few workgroups whose threads hold several
pairs in flight: planes of one pair to one more than a whole round of all of them
(32768 doubles), odd and even, bitwise in both directions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (nx + 2) (ny + 2) = 15, 513, 8190, 8192, 32767, 32768, 32769, 65536, 98307
@pytest.mark.parametrize("nx,ny", [(3, 1), (25, 17), (88, 89), (126, 62), (215, 149), (254, 126),
                                   (31, 991), (254, 254), (31, 2977)])
def test_planes_cross_unchanged(nx, ny):
    from fluidsim_amd import Discharge, configs

    d = Discharge(configs.base(nx, ny, grid_x=0))
    rng = np.random.default_rng(nx * ny)
    want = {(f, lev): rng.standard_normal((ny + 2, nx + 2)) for f in ("ni", "nm") for lev in (1, 2, 3)}
    for (f, lev), a in want.items():
        d.set(f, lev, a)
    for (f, lev), a in want.items():
        assert np.array_equal(d.get(f, lev), a), (f, lev)
    d.close()
