"""The walk over a query's cells loads the next step's photons ahead in a
session without a photon filter, and not in one with a filter nor in a batch.
The photons are visited in the same order, so a batch's image is its session's
bit for bit with every filter: cells of no photon, of fewer than a step's four,
and of many."""
import numpy as np
import pytest

from gpu_common import ctx, say, small_scene

import ppmpa_amd as P
from ppmpa_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,radius", [(1, 0.05), (40, 0.2), (3000, 0.01), (20000, 0.1)])
@pytest.mark.parametrize("pfilter", [A.FILTER_NONE, A.FILTER_CONE, A.FILTER_GAUSS])
def test_batch_image_is_the_session_image(n, radius, pfilter):
    say("walk forms", n, radius, pfilter)
    c = ctx()
    dss = [P.DeviceScene(c, small_scene("two_spheres", 56, 40)), P.DeviceScene(c, small_scene("caustic", 40, 33))]
    cfgs = [P.pass_cfg(seed=4 + i, n_photon=n + i, radius0=radius, alpha=2.0 / 3.0, max_depth=6, pfilter=pfilter,
                       use_classic=False, pipelines=2) for i in range(2)]
    b = P.Batch(c, dss, cfgs, [3, 3])
    b.run()
    for i in range(2):
        s = P.Session(c, dss[i], cfgs[i])
        s.run(3)
        assert np.array_equal(b.image(i)[0], s.image()[0])
        s.close()
    b.close()
