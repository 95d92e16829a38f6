"""Results that cross in slots of staging memory when they are to be stopped
(an overflow in the pass) and when the process may start no thread."""
import ctypes as C
import resource

import numpy as np
import pytest

from gpu_common import ctx, say

import ppmpa_amd as P
from ppmpa_amd import _abi as A
from ppmpa_amd import scene as S

pytestmark = pytest.mark.gpu

SLOT = (1 << 20) - 256
SIDES = {1: (160, 120), 4: (320, 230), 9: (512, 380)}  # slots of mean and variance: (width, height)


def _branching(w, h):
    """A box and eight spheres of a material that is shaded, reflects and
    refracts at every hit: 51 queries per pixel at depth 8, against 17 slots in
    place and two more per pixel of the picture."""
    sc = P.cornell_box(P.Scene())
    m = sc.add_material(S.simple((0.5,) * 3, (0.3,) * 3, 0.3, 0.0, 0.0, ior=(1.5,) * 3))
    for s in sc.shapes[:5]:
        s.material = m
    for i in range(8):
        sc.shapes.append(S.sphere((0.25 + 0.5 * (i & 1), 0.25 + 0.25 * (i & 2), 0.25 + 0.125 * (i & 4)), 0.21, m))
    sc.camera = S.box_camera(w, h)
    return sc


@pytest.mark.parametrize("slots", sorted(SIDES))
def test_overflow_writes_nothing(slots):
    w, h = SIDES[slots]
    say("staging stop", slots)
    assert -(-3 * w * h * 16 // SLOT) == slots
    c = ctx()
    cfg = P.pass_cfg(seed=1, n_photon=1000, radius0=0.05, alpha=2.0 / 3.0, max_depth=8)
    s = P.Session(c, P.DeviceScene(c, _branching(w, h)), cfg)
    s.run(1)
    for _ in range(3):
        mean, var = np.full((h, w, 3), 7.0), np.full((h, w, 3), 8.0)
        n = C.c_uint32()
        assert c.lib.ppm_session_image(s.h, mean.ctypes.data_as(A.dp), var.ctypes.data_as(A.dp),
                                       C.byref(n)) == A.PPM_E_RANGE
        assert b"overflow query slots" in c.lib.ppm_last_error(c.h)
        assert (mean == 7.0).all() and (var == 8.0).all()
    s.close()
    # the staging memory serves the next calls as before
    s = P.Session(c, P.DeviceScene(c, P.two_spheres_scene(w, h)), cfg)
    s.run(2)
    shared = s.image()[:2]
    s.close()
    other = P.Context(0)
    s = P.Session(other, P.DeviceScene(other, P.two_spheres_scene(w, h)), cfg)
    s.run(2)
    alone = s.image()[:2]
    other.close()
    assert np.array_equal(shared[0], alone[0]) and np.array_equal(shared[1], alone[1]) and alone[0].mean() > 0


def test_without_threads():
    """The same image from one thread, where no further one can be started."""
    say("staging without threads")
    w, h = SIDES[9]
    c = ctx()
    s = P.Session(c, P.DeviceScene(c, P.two_spheres_scene(w, h)),
                  P.pass_cfg(seed=1, n_photon=1000, radius0=0.05, alpha=2.0 / 3.0, max_depth=8))
    s.run(2)
    want = s.image()[:2]
    soft, hard = resource.getrlimit(resource.RLIMIT_NPROC)
    resource.setrlimit(resource.RLIMIT_NPROC, (1, hard))
    try:
        got = s.image()[:2]
    finally:
        resource.setrlimit(resource.RLIMIT_NPROC, (soft, hard))
    s.close()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
