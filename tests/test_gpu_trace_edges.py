"""The photon trace at the edges of its emission batches: a wave emits 64
photons at a time and hands them to lanes as they fall idle, over waves of up
to 256 photons each while there are few photons.  Every photon's walk depends
on its own random stream only, so the records of the first n photons are the
same bits however many are traced; the longest trace is checked against the
oracle elsewhere (test_gpu_trace.py)."""
import functools

import numpy as np
import pytest

from gpu_common import ctx, keyed_photons, say, small_scene

import ppmpa_amd as P
from ppmpa_amd import scene as S

pytestmark = pytest.mark.gpu

FULL = 9000


def _scene(kind):
    if kind == "box":
        return small_scene("caustic")
    sc = S.reference_room()  # TS surfaces: a bounce draws up to seven numbers
    if kind == "point":      # rejection: any number of draws at emission
        sc.lights = [S.point_light((1, 1, 1), 5.0, (0.0, 3.0, 2.5))]
    return sc


@functools.lru_cache(maxsize=None)
def _traced(kind, n):
    c = ctx()
    ds = P.DeviceScene(c, _scene(kind))
    pos, dir, wl, meta = P.trace_photons(c, ds, seed=3, pass_=2, n_photon=n, max_depth=9).download()
    return keyed_photons(meta, pos, dir, wl)


@pytest.mark.parametrize("kind", ["box", "room", "point"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 129, 256, 257, 1000, 4097])
def test_first_photons_the_same_for_any_count(kind, n):
    say("trace edges", kind, n)
    full, got = _traced(kind, FULL), _traced(kind, n)
    first = full[0] < n * 64  # key = photon * 64 + depth
    assert np.array_equal(full[0][first], got[0])
    for a, b in zip(full[1:], got[1:]):
        assert np.array_equal(a[first], b)
