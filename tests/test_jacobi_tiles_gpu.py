"""GPU: the Jacobi-PCG iteration's 64 x 8 tiles at grids that end inside a tile,
along either axis, and with several tiles per workgroup (more than 1024).  The
solver's recurrence reaches 1e-8; the residual recomputed from the system
differs from it by rounding (some 1e-13 a step at most over these solves)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,cyl", [(513, 9, 0), (65, 71, 1), (3, 800, 0), (200, 137, 0),
                                       (64, 512, 1), (1030, 521, 0)])
def test_jacobi_solve_reaches_the_tolerance(nx, ny, cyl):
    from fluidsim_amd import Discharge, configs

    d = Discharge(configs.base(nx, ny, volts=200.0, rtol=1e-8, solver=0, cyl=cyl, grid_x=0))
    d.init_gaussian(seed=nx)
    lerr, st = d.lapl_solve()
    assert lerr == 0 and 0 < st.iters < 20000
    assert st.resid <= 1.01e-8
    print((nx, ny), st.iters, st.resid)
