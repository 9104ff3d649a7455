"""GPU: evaluations from several threads at once, which share the device's staging
array or, when it is taken and the call is large (from 8192 fluxes), allocate."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 16, 17, 100), (8191, 8192, 32768, 32769),
                                   (3, 32768, 8192, 20000)])
def test_threads_get_their_own_results(sizes):
    from fluidsim_amd import eval_fits, eval_flux

    rng = np.random.default_rng(len(sizes) + sizes[0])
    a = [10.0 ** rng.uniform(-2, 2, (n, 7)) for n in sizes]
    want = [(eval_flux(x), eval_fits(x[:, 0])) for x in a]

    def work(i):
        return [(eval_flux(a[i]), eval_fits(a[i][:, 0])) for _ in range(30)]

    with ThreadPoolExecutor(len(sizes)) as ex:
        for (flux, fits), got in zip(want, ex.map(work, range(len(sizes)))):
            for f, t in got:
                assert np.array_equal(f, flux) and np.array_equal(t, fits)
