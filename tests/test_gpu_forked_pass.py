"""A session or batch of one pipeline runs the eye branch of its pass graphs
beside the photon branch, the two sharing no memory.  The passes are those of
the same session without graphs, whose pass is one chain, bit for bit: over many
replays, with runs in pieces, other work on the device between them, a reset, a
backward and a change of the tile shape."""
import numpy as np
import pytest

from gpu_common import ctx, say

import ppmpa_amd as P

pytestmark = pytest.mark.gpu

NO_GRAPH = 2


def _scene(kind):
    if kind == "tree":
        return P.mesh_scene(72, 56, subdiv=2, n_spheres=20, seed=3)
    return P.caustic_scene(*kind)


def _cfg(n, flags=0):
    return P.pass_cfg(seed=6, n_photon=n, radius0=0.03, alpha=2.0 / 3.0, max_depth=7, pipelines=1, flags=flags)


@pytest.mark.parametrize("kind,n", [((9, 7), 1), ((64, 48), 3000), ((200, 150), 60000), ((640, 480), 300000),
                                    ("tree", 20000)])
def test_session_equals_one_chain(kind, n):
    say("forked pass", kind, n)
    c = ctx()
    ds, other = P.DeviceScene(c, _scene(kind)), P.DeviceScene(c, P.two_spheres_scene(96, 64))
    forked, chain = P.Session(c, ds, _cfg(n)), P.Session(c, ds, _cfg(n, NO_GRAPH))
    between = P.Session(c, other, P.pass_cfg(seed=1, n_photon=30000, radius0=0.03, alpha=2.0 / 3.0, max_depth=6))
    for s in (forked, chain):
        for k in (1, 4, 2):
            s.run(k)
            between.run(3)
    want = chain.image()
    got = forked.image()
    assert got[2] == want[2] == 7 and want[0].any()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    g = np.ones_like(want[0])
    a, b = forked.backward(g), chain.backward(g)
    assert np.allclose(a[0], b[0], rtol=1e-5, atol=1e-9 * max(1e-30, np.abs(b[0]).max()))
    for s in (forked, chain):
        s.set_tile_width(16)
        s.reset()
        s.run(5)
    got, want = forked.image(), chain.image()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    for s in (forked, chain, between):
        s.close()


@pytest.mark.parametrize("sides", [(40,), (33, 64, 120)])
def test_batch_of_one_pipeline_equals_sessions(sides):
    say("forked batch", sides)
    c = ctx()
    dss = [P.DeviceScene(c, P.caustic_scene(s, s - 3)) for s in sides] + [P.DeviceScene(c, _scene("tree"))]
    cfgs = [_cfg(2000 * (i + 1)) for i in range(len(dss))]
    n = [5 - i for i in range(len(dss))]
    b = P.Batch(c, dss, cfgs, n)
    b.run(2)
    b.run()
    for i, ds in enumerate(dss):
        s = P.Session(c, ds, cfgs[i])
        s.run(n[i])
        got, want = b.image(i), s.image()
        # equal but for pixels with overflowed queries (added with atomics)
        assert np.allclose(got[0], want[0], rtol=1e-6, atol=0.0) and (got[0] == want[0]).mean() >= 0.99
        s.close()
    b.close()
