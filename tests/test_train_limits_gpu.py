"""GPU: a training batch that the loss partials have no room for is refused
before anything is sized by it, and changes nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [32769, 2**31 - 1])  # 2^27 pixels fit: 32768 of 64 x 64
def test_too_large_a_batch_is_refused(batch):
    from fluidsim_amd import Discharge, configs
    from fluidsim_amd.learn import LearnedPreconditioner
    from fluidsim_amd.lib import FsError

    d = Discharge(configs.config1(128))
    d.init_gaussian(seed=1)
    out = []
    for refused in (False, True):
        net = LearnedPreconditioner(20, 64, 64, seed=3)
        net.harvest(d)
        if refused:
            before = net.weights()
            with pytest.raises(FsError, match="batch too large"):
                net.train(100, batch=batch, lr=1e-3, seed=5)
            assert np.array_equal(net.weights(), before)
            assert net.train(0, batch=batch).size == 0
        out.append((np.asarray(net.train(3, batch=4, lr=1e-3, seed=5)), net.weights()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
