"""GPU: training steps are enqueued in rounds of 64; a call of many steps gives,
bit for bit, the losses and weights of as many calls of one step, across the
end of a round and for batches whose partial sums outgrow the first buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GAMMA = 0x9E3779B97F4A7C15  # the batch indices' generator advances by this per sample


@pytest.mark.parametrize("steps,batch", [(1, 1), (66, 3), (129, 2), (2, 40)])
def test_rounds_equal_single_steps(steps, batch):
    from fluidsim_amd import Discharge, configs
    from fluidsim_amd.learn import LearnedPreconditioner

    d = Discharge(configs.config1(128))
    d.init_gaussian(seed=1)
    out = []
    for single in (False, True):
        net = LearnedPreconditioner(20, 64, 64, seed=3)
        net.harvest(d)
        if single:
            loss = [net.train(1, batch=batch, lr=1e-3, seed=(5 + k * batch * GAMMA) % 2**64)[0]
                    for k in range(steps)]
        else:
            loss = net.train(steps, batch=batch, lr=1e-3, seed=5)
        out.append((np.asarray(loss), net.weights()))
    assert np.all(np.isfinite(out[0][0]))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
