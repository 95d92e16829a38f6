"""The photon trace emits 64 photons at a time through LDS in scenes without a
small tree and on demand in scenes with one.  The records are the same bits
either way: a room of spheres traced with its tree and as a list, at the edges
of the emission batches and of the tracing waves' shares."""
import numpy as np
import pytest

from gpu_common import ctx, keyed_photons, say

import ppmpa_amd as P
from ppmpa_amd import _abi as A

pytestmark = pytest.mark.gpu


def _room(kind):
    rng = np.random.default_rng(11)
    sc = P.cornell_box(P.Scene())
    mats = [sc.add_material(P.lambertian(0.7)), sc.add_material(P.mirror()), sc.add_material(P.glass(1.5))]
    for i in range(5):
        for j in range(4):
            for k in range(5):
                c = (np.array([i, j, k]) + 0.5) / 5 * 0.9 + 0.05
                sc.shapes.append(P.sphere(tuple(c), float(rng.uniform(0.02, 0.07)), mats[int(rng.integers(0, 3))]))
    if kind == "point":  # rejection: any number of draws at emission
        from ppmpa_amd.scene import point_light
        sc.lights = [point_light((1, 1, 1), 5.0, (0.5, 0.95, 0.5))]
    sc.camera = P.pinhole(32, 24, (0.5, 0.5, -0.87), (0.5, 0.5, 1.0), 60.0)
    return sc


@pytest.mark.parametrize("kind", ["panel", "point"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 4097, 60001])
def test_records_with_and_without_the_tree(kind, n):
    say("trace trees", kind, n)
    c = ctx()
    got = []
    for flag in (A.SCENE_BVH_ON, A.SCENE_BVH_OFF):
        sc = _room(kind)
        sc.bvh = flag
        ds = P.DeviceScene(c, sc)
        assert (ds.stats()[1] > 0) == (flag == A.SCENE_BVH_ON)
        pos, dir, wl, meta = P.trace_photons(c, ds, seed=3, pass_=2, n_photon=n, max_depth=9).download()
        got.append(keyed_photons(meta, pos, dir, wl))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
