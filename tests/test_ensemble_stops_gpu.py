"""GPU: ensembles whose multigrid launches cover more bands than the card holds
workgroups at once, with solves that stop at different iterations: a workgroup
then goes on from a member that has stopped to one that has not, and may start
after another has recorded that a member stopped.  Members end bitwise where
their solo runs do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bands(c):  # 32 x 16 cells each on the finest level
    return -(-c["nx"] // 32) * -(-c["ny"] // 16)


def _compare(cfgs, passes):
    """Logs of the members after `passes`, their state compared with solo runs."""
    from fluidsim_amd import Discharge
    from fluidsim_amd.ensemble import Ensemble

    E = Ensemble(cfgs)
    for m, c in zip(E.members, cfgs):
        m.init_gaussian(seed=c["seed"])
    E.run(passes)
    logs = []
    for i, (m, c) in enumerate(zip(E.members, cfgs)):
        d = Discharge(c)
        d.init_gaussian(seed=c["seed"])
        d.run(passes)
        for f in ("ni", "ne", "nt", "nm", "ph"):
            assert np.array_equal(m.get(f), d.get(f)), (i, c["nx"], c["ny"], f)
        assert np.array_equal(m.log(), d.log()), i
        assert m.scalars() == d.scalars(), i
        logs.append(m.log())
        d.close()
    E.close()
    return logs


def test_members_that_stop_at_different_iterations():
    from fluidsim_amd import configs

    cfgs = configs.config3(24, base_seed=2, lo=150, hi=260, warm=0)
    assert sum(map(_bands, cfgs)) > 2 * 768  # ranges of several bands, across members
    for i, c in enumerate(cfgs):
        c["lapl_rtol"] = 10.0 ** (-2 - i % 9)
    logs = _compare(cfgs, 8)
    iters = [int(r[7]) for log in logs for r in log if r[6] >= 0]
    assert len(set(iters)) > 4, sorted(set(iters))


def test_warm_starts_that_meet_the_tolerance():
    """Solves that the initial test ends (0 iterations) still form their warm
    start on every band, in launches of more bands than workgroups fit (1024)."""
    from fluidsim_amd import configs

    cfgs = configs.config3(24, base_seed=4, lo=150, hi=260, warm=2)
    assert sum(map(_bands, cfgs)) > 1024
    for c in cfgs:
        c["lapl_rtol"] = 1e-2
    logs = _compare(cfgs, 14)
    zero = sum(int(r[7] == 0) for log in logs for r in log if r[6] >= 0)
    print("solves ended by the initial test:", zero)
    assert zero > 24
