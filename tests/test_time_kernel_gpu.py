"""GPU: fs_time_kernel's ids."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,ids", [(96, 80, (0, 6, 15, 19, 22, 41, 60, 99)),
                                       (4, 4, (13, 17, 18, 20, 40))])
def test_a_refused_id_leaves_the_handle_as_it_was(nx, ny, ids):
    """(A timed id runs with the tolerance 0 and 2^30 iterations, and puts the
    caller's settings back.)"""
    from fluidsim_amd import Discharge, configs
    from fluidsim_amd.lib import FsError

    out = []
    for refused in (False, True):
        d = Discharge(configs.base(nx, ny, volts=200.0, rtol=1e-6, maxit=500, grid_x=0))
        d.init_gaussian(seed=1)
        if refused:
            for k in ids:
                with pytest.raises(FsError):
                    d.time_kernel(k, 2)
        lerr, st = d.lapl_solve()
        assert lerr == 0
        out.append((st.iters, st.resid, d.get("ph")))
        d.close()
    assert out[0][:2] == out[1][:2]
    assert np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("nx,ny,first", [(96, 80, [0]), (512, 512, [0]), (1024, 512, [0, 1]),
                                         (300, 200, [0])])
def test_up_ids_are_the_launches_of_an_iteration(nx, ny, first):
    """The up step of a level of at most 512 tiles of 32 x 16 cells comes with
    those of the one or two tile levels below it; only the launches there are
    have a time."""
    from fluidsim_amd import Discharge, configs
    from fluidsim_amd.lib import FsError

    d = Discharge(configs.base(nx, ny, volts=200.0, grid_x=0))
    d.init_gaussian(seed=1)
    d.lapl_solve()
    got = []
    for lvl in range(6):
        try:
            assert d.time_kernel(40 + lvl, 4) > 0.0
            got.append(lvl)
        except FsError as e:
            assert "above" in str(e) or "no tile kernel" in str(e)
    assert got == first
    assert d.time_kernel(14, 4) > 0.0 and d.time_kernel(17, 4) > 0.0
    d.close()
