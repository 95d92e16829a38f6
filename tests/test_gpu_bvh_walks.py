"""Walks of large trees, which the lanes of a tracing or eye wave share: a lane
without work takes a subtree that another put off.  A photon's records do not
depend on which other photons its wave holds, down to a single one (63 helpers)
and the ends of the emission batches; and batches whose rooms hold large trees,
small ones (walked lane by lane, from LDS) and none, in one launch."""
import functools

import numpy as np
import pytest

from gpu_common import ctx, keyed_photons, say

import oracle_lib as O
import ppmpa_amd as P

pytestmark = pytest.mark.gpu

FULL = 5000


def _mesh(side=40):
    return P.mesh_scene(side, side, subdiv=3, n_spheres=12, seed=4)  # 1292 primitives


@functools.lru_cache(maxsize=None)
def _traced(n):
    c = ctx()
    ds = P.DeviceScene(c, _mesh())
    assert ds.stats()[1] > 512  # past the trees that are copied to LDS
    pos, dir, wl, meta = P.trace_photons(c, ds, seed=3, pass_=2, n_photon=n, max_depth=9).download()
    return keyed_photons(meta, pos, dir, wl)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 257, 1000])
def test_photons_the_same_for_any_count(n):
    say("mesh trace", n)
    full, got = _traced(FULL), _traced(n)
    first = full[0] < n * 64  # key = photon * 64 + depth
    assert np.array_equal(full[0][first], got[0])
    for a, b in zip(full[1:], got[1:]):
        assert np.array_equal(a[first], b)


@pytest.mark.parametrize("depth", [1, 2, 10])
def test_mesh_pass_matches_oracle(depth):
    """As the smoke check of a pass: FP32 walks against the FP64 oracle."""
    say("mesh pass", depth)
    sc = _mesh()
    cfg = P.pass_cfg(seed=1, n_photon=20000, radius0=0.03, alpha=2.0 / 3.0, max_depth=depth)
    c = ctx()
    mean, _, _ = P.run_passes(c, P.DeviceScene(c, sc), cfg, 1)
    omean = O.OScene(sc).run_passes(cfg, 1)[0]
    assert abs(mean.mean() - omean.mean()) <= 2e-3 * omean.mean()
    close = (np.abs(mean - omean) <= 1e-3 * np.maximum(np.abs(omean), 1e-3 * np.abs(omean).max())).all(axis=2)
    assert close.mean() > 0.95


@pytest.mark.parametrize("kinds", ["L", "LS", "LN", "SN", "LSN"])
def test_mixed_batch_equals_sessions(kinds):
    """L: a room with a large tree, S: with a small one, N: without."""
    say("mixed batch", kinds)
    c = ctx()
    small = [x[0] for x in P.batch_scenes(n=40, seed=5, max_side=40, min_side=32) if len(x[0].shapes) - 6 >= 80][0]
    scenes = {"L": _mesh(), "S": small, "N": P.two_spheres_scene(40, 40)}
    dss = [P.DeviceScene(c, scenes[k]) for k in kinds]
    cfgs = [P.pass_cfg(seed=7 + i, n_photon=6000 + 501 * i, radius0=0.03, alpha=2.0 / 3.0, max_depth=8, pipelines=2)
            for i in range(len(kinds))]
    b = P.Batch(c, dss, cfgs, [3] * len(kinds))
    b.run()
    for i, (ds, cfg) in enumerate(zip(dss, cfgs)):
        s = P.Session(c, ds, cfg)
        s.run(3)
        m, v, _ = s.image()
        bm, bv, _ = b.image(i)
        # equal but for pixels with overflowed queries (added with atomics)
        assert np.allclose(bm, m, rtol=1e-6, atol=0.0) and (bm == m).mean() >= 0.99
        assert np.allclose(bv, v, rtol=1e-5, atol=1e-12)
        s.close()
    b.close()
