"""The mean and variance of a session's passes, merged on the device from the
pipelines' sums and brought to the host in chunks: equal, bit for bit, to the
same double operations in numpy on the passes' own images, for images below,
at and beyond a chunk of the staging memory (2^19 - 32 values with the mean
alone, half as many with the variance)."""
import numpy as np
import pytest

from gpu_common import ctx, say, small_scene

import ppmpa_amd as P

pytestmark = pytest.mark.gpu


def _cfg(first, pipelines):
    return P.pass_cfg(seed=5, n_photon=2000, radius0=0.05, alpha=2.0 / 3.0, max_depth=5, first_pass=first,
                      pipelines=pipelines)


@pytest.mark.parametrize("pipelines", [1, 2, 4])
@pytest.mark.parametrize("w,h", [(1, 1), (31, 17), (256, 341), (254, 344), (431, 607), (512, 342)])
def test_mean_and_variance(w, h, pipelines):
    say("image", w, h, pipelines)
    c = ctx()
    ds = P.DeviceScene(c, small_scene("caustic", w, h))
    passes = []
    for k in range(3):
        s = P.Session(c, ds, _cfg(k + 1, 1))
        s.run(1)
        passes.append(s.image(False)[0])
        s.close()
    s = P.Session(c, ds, _cfg(1, pipelines))
    s.run(3)
    mean, var, n = s.image()
    alone, none, _ = s.image(False)
    s.close()
    assert n == 3 and none is None and np.array_equal(mean, alone)
    # each pipeline adds its passes in order; the pipelines are added in order
    add = [sum((passes[k] for k in range(j, 3, pipelines)), np.zeros_like(mean)) for j in range(pipelines)]
    sq = [sum((passes[k] * passes[k] for k in range(j, 3, pipelines)), np.zeros_like(mean)) for j in range(pipelines)]
    t, q = sum(add, np.zeros_like(mean)), sum(sq, np.zeros_like(mean))
    assert np.array_equal(mean, t / 3.0)
    assert np.array_equal(var, np.maximum(0.0, (q - t * t / 3.0) / 2.0))
