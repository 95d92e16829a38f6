"""run_passes, which knows its passes and takes no more sets of buffers than
they need: image, variance and counts of a session that runs as many, bit for
bit, from none to more than the pipelines, for every number of pipelines, and
the same error for a refused configuration."""
import numpy as np
import pytest

from gpu_common import ctx, say, small_scene

import ppmpa_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pipelines", [0, 1, 3])
@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 5, 9])
def test_equals_a_session(n, pipelines):
    say("run_passes", n, pipelines)
    c = ctx()
    ds = P.DeviceScene(c, small_scene("two_spheres", 61, 45))
    cfg = P.pass_cfg(seed=8, n_photon=5000, radius0=0.04, alpha=2.0 / 3.0, max_depth=7, pipelines=pipelines)
    mean, var, t = P.run_passes(c, ds, cfg, n)
    s = P.Session(c, ds, cfg)
    s.run(n)
    m, v, k = s.image()
    u = s.timings()
    s.close()
    assert k == n and np.array_equal(mean, m) and np.array_equal(var, v)
    for key in ("passes", "photons_emitted", "photons_stored", "gather_queries"):
        assert t[key] == u[key], key
    assert (n == 0) == (not mean.any())


def test_refuses_as_a_session():
    c = ctx()
    ds = P.DeviceScene(c, small_scene("two_spheres", 16, 16))
    cfg = P.pass_cfg(seed=8, n_photon=0, radius0=0.04, alpha=2.0 / 3.0, max_depth=7)
    errs = []
    for f in (lambda: P.run_passes(c, ds, cfg, 1), lambda: P.Session(c, ds, cfg)):
        with pytest.raises(P.PpmError) as e:
            f()
        errs.append((e.value.status, str(e.value)))
    assert errs[0] == errs[1]
