"""Axis-aligned rectangles of the shape list are tested without the products
by their sides' zero components.  The scene's BVH tests the same shapes with
the general parallelogram test, so the two forms of one scene must report the
same distances and shapes, bit for bit, for every orientation and order of
the sides, sides of either sign, and rays along the axes, in the plane, from
the plane and through corners and edges."""
import numpy as np
import pytest

from gpu_common import ctx, say

import ppmpa_amd as P
from ppmpa_amd import _abi as A
from ppmpa_amd import scene as S

pytestmark = pytest.mark.gpu


def _rects(i, j, rng):
    """Rectangles with sides along axis i, then axis j."""
    out = []
    for si in (1.0, -0.37):
        for sj in (0.8, -1.0):
            p = np.round(rng.uniform(-1.0, 1.0, 3), 3)
            e1, e2 = np.zeros(3), np.zeros(3)
            e1[i], e2[j] = si, sj
            out.append((p, e1, e2))
    p, e1, e2 = np.zeros(3), np.zeros(3), np.zeros(3)  # at the origin, unit sides
    e1[i] = e2[j] = 1.0
    return out + [(p, e1, e2)]


def _scene(rects, flags):
    sc = S.Scene()
    m = sc.add_material(S.lambertian(0.5))
    sc.shapes += [S.parallelogram(tuple(p), tuple(p + a), tuple(p + b), m) for p, a, b in rects]
    # far apart, so that no rectangle is wide against the scene
    sc.shapes += [S.sphere((40.0, 40.0, 40.0), 0.5, m), S.sphere((-40.0, -40.0, -40.0), 0.5, m)]
    sc.lights.append(S.point_light((1, 1, 1), 1.0, (0, 30, 0)))
    sc.camera = S.box_camera(8, 8)
    sc.bounds_min, sc.bounds_max = (-41, -41, -41), (41, 41, 41)
    sc.bvh = flags
    return sc


@pytest.mark.parametrize("i,j", [(0, 1), (0, 2), (1, 0), (1, 2), (2, 0), (2, 1)])
def test_rectangle_equals_the_general_test(i, j):
    say("rect", i, j)
    rng = np.random.default_rng(10 * i + j)
    rects = _rects(i, j, rng)
    o, d = [rng.uniform(-2, 2, (20000, 3))], [rng.normal(size=(20000, 3))]
    for p, a, b in rects:
        uv = np.array([(0, 0), (1, 0), (0, 1), (1, 1), (0.5, 0), (0, 0.5), (0.5, 0.5), (1, 0.25), (0.25, 1)])
        x = p + uv[:, :1] * a + uv[:, 1:] * b
        n = np.cross(a, b)
        for off in (n, -n, 1e-3 * n, a + n, b - n, a, b, 0 * n):  # towards, in and from the plane
            o.append(x + off)
            d.append(np.where(np.abs(off).sum() > 0, -off, n) * np.ones_like(x))
        o.append(x)
        d.append(rng.normal(size=x.shape))
    for axis in range(3):  # along the axes: two zero components, of either sign
        for s in (1.0, -1.0):
            e = np.full((500, 3), 0.0 if s > 0 else -0.0)
            e[:, axis] = s
            o.append(rng.uniform(-1.5, 1.5, (500, 3)))
            d.append(e)
    o, d = np.concatenate(o), np.concatenate(d)
    c = ctx()
    lst, tree = (P.DeviceScene(c, _scene(rects, f)) for f in (A.SCENE_BVH_OFF, A.SCENE_BVH_ON))
    assert lst.stats()[1] == 0 and tree.stats()[1] == len(rects) + 2
    t0, k0 = lst.intersect(o, d)
    t1, k1 = tree.intersect(o, d)
    assert (k0 >= 0).sum() > 1000
    assert np.array_equal(k0, k1) and np.array_equal(t0, t1)
