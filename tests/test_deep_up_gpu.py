"""GPU: a solo handle makes the up steps of two or three multigrid levels in one
launch where the finest of them has at most 512 tiles; an ensemble keeps a launch
per level.
Members end bitwise where their solo runs do, on grids of two to four tile levels
with odd sides, tile remainders and levels on both sides of the limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("warm", [0, 1])
def test_members_equal_their_solo_runs_bitwise(warm):
    from fluidsim_amd import Discharge, configs
    from fluidsim_amd.ensemble import Ensemble

    sizes = [(129, 130), (300, 200), (70, 600), (513, 95), (257, 512), (512, 256), (514, 257),
             (601, 433), (1025, 300)]
    # (the widest on the uniform 5 cm grid: its cells on 1 cm would be too small
    # for the time step's lower limit)
    cfgs = [configs.base(nx, ny, volts=250.0, p_torr=2.0, ratio_x=1.05 ** (64.0 / nx), warm=warm)
            if nx < 1000 else dict(configs.config2(nx, warm=warm), ny=ny) for nx, ny in sizes]
    E = Ensemble(cfgs)
    for i, m in enumerate(E.members):
        m.init_gaussian(seed=i)
    E.run(5)
    for i, (m, c) in enumerate(zip(E.members, cfgs)):
        d = Discharge(c)
        d.init_gaussian(seed=i)
        d.run(5)
        for f in ("ni", "ne", "nt", "nm", "ph"):
            assert np.array_equal(m.get(f), d.get(f)), (sizes[i], f)
        assert np.array_equal(m.log(), d.log()), sizes[i]
        d.close()
    E.close()
