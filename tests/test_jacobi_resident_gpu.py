"""GPU: Jacobi-PCG solves with more workgroups than the card holds at once (a
launch of 1024 workgroups of eight waves).  Late workgroups must take the same
decision as the first: the potential ends on the solution of the assembled
system, recomputed here from its rows, and stays as it was where the solve does
not converge."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _residual(b, A5, x):
    """b + A x in reference form (rows W, E, S, N, C); the solve leaves it at
    rtol |b|."""
    p = np.pad(x, 1)
    W, E, S, N, C = (A5[..., k] for k in range(5))
    return (b + W * p[1:-1, :-2] + E * p[1:-1, 2:] + S * p[:-2, 1:-1] + N * p[2:, 1:-1] +
            C * x)


@pytest.mark.parametrize("nx,ny", [(1024, 513), (700, 811)])
def test_solution_of_the_assembled_system(nx, ny):
    from fluidsim_amd import Discharge, configs

    rtol = 1e-6
    cfg = configs.base(nx, ny, volts=200.0, rtol=rtol, solver=0, debug=1, grid_x=0)
    d = Discharge(cfg)
    d.init_gaussian(seed=1)
    b, A5 = d.lapl_assemble()
    ph0 = d.get("ph")[1:-1, 1:-1]
    lerr, st = d.lapl_solve()
    assert lerr == 0 and 0 < st.iters < 20000
    ph = d.get("ph")[1:-1, 1:-1]
    x = ph - ph0
    rel = np.linalg.norm(_residual(b, A5.reshape(ny, nx, 5), x)) / np.linalg.norm(b)
    # what the subtraction ph - ph0 loses enters each row as at most 8 C eps |ph|
    # (four neighbours' coefficients sum to C)
    lost = 8.0 * np.finfo(float).eps * np.linalg.norm(A5[..., 4].ravel()) * np.abs(ph).max()
    print((nx, ny), st.iters, st.resid, rel, lost / np.linalg.norm(b))
    assert rel <= 1.01 * rtol + lost / np.linalg.norm(b)
    d.close()


@pytest.mark.parametrize("nx,ny", [(257, 2), (1000, 3), (1500, 4), (1500, 5), (513, 8)])
def test_thin_grids(nx, ny):
    """Tiles of four rows where the grid has no more, of eight above."""
    test_solution_of_the_assembled_system(nx, ny)


def test_unconverged_solve_leaves_the_potential():
    from fluidsim_amd import Discharge, configs

    d = Discharge(configs.base(1024, 513, volts=200.0, solver=0, maxit=40, grid_x=0))
    d.init_gaussian(seed=1)
    ph0 = d.get("ph")
    lerr, st = d.lapl_solve()
    assert lerr == 1 and st.iters == 40
    assert np.array_equal(d.get("ph"), ph0)
    d.close()
