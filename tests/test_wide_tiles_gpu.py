"""GPU: the tiles of the stage and assembly kernels with more waves than cells,
which launches of few tiles take, at the edges of their shapes (one row, one
column, remainders) and on both sides of the limit of 256 tiles.  The 64 x 4
stage tiles give the bits of the 64 x 8 ones; the assembly is compared with the
oracle on the same state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cfg(nx, ny, **kw):
    from fluidsim_amd import configs

    return configs.base(nx, ny, volts=250.0, ratio_x=1.05 ** (64.0 / max(nx, 16)), **kw)


@pytest.mark.parametrize("nx,ny,kw", [(3, 2, {}), (64, 4, {}), (65, 5, dict(cyl=1)),
                                      (130, 33, dict(rwall=1)), (40, 1, {}), (64, 1024, {}),
                                      (64, 1025, {}), (513, 113, {})])
def test_stage_tiles(nx, ny, kw):
    from fluidsim_amd import Discharge

    out = []
    for ty in (4, 8):
        d = Discharge(_cfg(nx, ny, stage_tile=ty, **kw))
        d.init_gaussian(seed=2)
        d.run(5)
        out.append([d.get(f, lev) for f in ("ni", "ne", "nt", "nm") for lev in (1, 2, 3)] +
                   [d.get("ph"), d.log()])
        d.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,ny", [(3, 2), (64, 8), (65, 9), (40, 31), (64, 2048), (64, 2049)])
def test_assembly(O, nx, ny):
    """(the tolerances of the assembly's parity test)"""
    from fluidsim_amd import Discharge

    cfg = _cfg(nx, ny, debug=1)
    d = Discharge(cfg)
    d.init_gaussian(seed=2)
    d.run(4)
    o = O.Oracle(dict(cfg, rtol=1e-13, maxit=20000, solver=0, nthreads=1))
    for f in ("ni", "ne", "nt", "nm"):
        o.set(f, 1, d.get(f, 1))
    o.set("ph", 1, d.get("ph"))
    o.set_scalars(d.scalars())
    b, A5 = d.lapl_assemble()
    st, b_o, A_o = o.lapl_assemble()
    assert st == 0
    assert np.linalg.norm(b - b_o) <= 1e-10 * np.linalg.norm(b_o)
    for c in range(5):
        assert np.linalg.norm(A5[..., c] - A_o[..., c]) <= 1e-12 * np.linalg.norm(A_o[..., c]), c
