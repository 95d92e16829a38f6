"""Buffers that outlive a call or a pass: the context's block that single
calls lay their buffers out in, and a session's pipelines after a reset.
Results equal, bit for bit, those of a context or session that has run
nothing else."""
import numpy as np
import pytest

from gpu_common import ctx, random_photons, say, small_scene

import ppmpa_amd as P

pytestmark = pytest.mark.gpu


def _eye(c, w, h, depth, seed):
    ds = P.DeviceScene(c, small_scene("caustic", w, h))
    ph = P.PhotonSet(c, 5000)
    ph.upload(*random_photons(5000, seed))
    m = P.build_photonmap(c, ph, 1e-3)
    return P.trace_eye(c, ds, m, seed, 1, 0.02 ** 2, max_depth=depth)


def _classic(c, w, h):
    return P.trace_classic(c, P.DeviceScene(c, small_scene("caustic", w, h)), 3, 1, (0.1, 0.1, 0.1))


def test_calls_of_different_sizes_share_the_block():
    say("workspace: eye and classic passes of different sizes in turn")
    calls = [lambda c: _eye(c, 40, 30, 4, 1), lambda c: _classic(c, 97, 61), lambda c: _eye(c, 200, 150, 16, 2),
             lambda c: _classic(c, 16, 9), lambda c: _eye(c, 40, 30, 4, 1), lambda c: _eye(c, 7, 5, 1, 3)]
    shared = [f(ctx()) for f in calls]
    for k, f in enumerate(calls):
        c = P.Context(0)
        alone = f(c)
        c.close()
        assert np.array_equal(shared[k], alone), k


@pytest.mark.parametrize("pipelines", [0, 1, 2, 3])
def test_reset_session_renders_as_a_new_one(pipelines):
    say("workspace: reset", pipelines)
    c = ctx()
    ds = P.DeviceScene(c, small_scene("caustic", 40, 30))

    def cfg():
        return P.pass_cfg(seed=9, n_photon=3000, radius0=0.05, alpha=2.0 / 3.0, max_depth=6, pipelines=pipelines)

    s = P.Session(c, ds, cfg())
    s.run(5)
    first = s.image()[0]
    for scale in (1.0, 0.5, 0.5, 2.0):
        ds.set_params(light_scale=scale)
        s.reset()
        s.run(2)
        s.run(3)
        mean, var, n = s.image()
        fresh = P.Session(c, ds, cfg())
        fresh.run(5)
        m2, v2, n2 = fresh.image()
        fresh.close()
        assert n == n2 == 5
        assert np.array_equal(mean, m2) and np.array_equal(var, v2)
        if scale == 1.0:
            assert np.array_equal(mean, first)
    s.close()
