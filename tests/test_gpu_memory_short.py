"""Calls while little device memory is free: photon sets of another context
hold the rest, as a framework beside the library would."""
import ctypes as C

import numpy as np
import pytest

from gpu_common import ctx, random_photons, say

import ppmpa_amd as P
from ppmpa_amd import _abi as A

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def _free():
    """The device's free memory, from the HIP runtime that the library is
    linked to (torch, once imported, brings another)."""
    free, total = C.c_size_t(), C.c_size_t()
    assert A.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


class _Rest:
    """The device's free memory, taken but for what leave() says."""

    def __enter__(self):
        self.c, self.mem = P.Context(0), []
        return self

    def leave(self, n):
        for step in (16 * GIB, GIB, GIB // 16):
            while _free() >= n + step:
                self.mem.append(P.PhotonSet(self.c, (step - (1 << 20)) // 32))  # 32 B per photon
        say("memory left: %.2f GiB" % (_free() / GIB))

    def __exit__(self, *exc):
        self.c.close()


def _session(c, ds, n_pass=7, backward=False):
    free = _free()
    s = P.Session(c, ds, P.pass_cfg(seed=5, n_photon=250_000, radius0=0.01, alpha=2 / 3, max_depth=16))
    took = free - _free()
    s.run(n_pass - 4)
    s.run(4)
    out = s.image()[:2]
    if backward:
        out += s.backward(np.ones_like(out[0]))
    s.close()
    return took, out


def test_automatic_session_gives_the_same_image():
    """A set of buffers takes 1.3 GiB here: four of them where memory is
    plenty, two where 8 GiB are free, one where 2.5 GiB are, whatever the
    context's idle block (up to 2 GiB) adds.  Image and variance are the same
    to the last bit; the adjoint adds floats by atomics in any order, up to
    some 160 of them to a photon: 160 * 2^-24."""
    say("memory short: automatic session")
    c = ctx()
    ds = P.DeviceScene(c, P.two_spheres_scene(512, 512))
    many, plenty = _session(c, ds, backward=True)
    again, same = _session(c, ds)
    assert np.array_equal(plenty[0], same[0]) and np.array_equal(plenty[1], same[1])
    with _Rest() as rest:
        for n, most in ((8 * GIB, 0.6), (5 * GIB // 2, 0.35)):
            rest.leave(n)
            few, short = _session(c, ds, backward=True)
            assert np.array_equal(plenty[0], short[0]) and np.array_equal(plenty[1], short[1])
            assert np.allclose(plenty[2], short[2], rtol=1e-5, atol=1e-9 * np.abs(plenty[2]).max())
            assert abs(plenty[3] - short[3]) <= 1e-12 * abs(plenty[3])
            assert few < most * many, (few, many)


def test_idle_block_is_given_back():
    """The block that a context keeps from an image of the classic tracer (over
    1 GiB) makes room for double positions (0.9 GiB) that the rest of the
    memory does not hold; the next image allocates it again."""
    say("memory short: idle block")
    c = P.Context(0)
    ds = P.DeviceScene(c, P.two_spheres_scene(1280, 720))
    ph = P.PhotonSet(c, 40_000_000)
    free = _free()
    img = P.trace_classic(c, ds, 3, 1)
    assert GIB < free - _free() <= 2 * GIB + GIB // 64, (free - _free()) / GIB
    rng = np.random.default_rng(1)
    pos, d = rng.random((500, 3)), rng.standard_normal((500, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    with _Rest() as rest:
        rest.leave(GIB // 2)
        ph.upload(pos, d, np.zeros(500, np.uint8))
    m = P.build_photonmap(c, ph, 1e-3)
    got = m.within(pos[:20], 0.2 ** 2, refine64=True)
    for q, i in zip(pos[:20], got):
        assert np.array_equal(i, np.nonzero(((pos - q) ** 2).sum(1) <= 0.2 ** 2)[0])
    assert np.array_equal(P.trace_classic(c, ds, 3, 1), img)
    c.close()


@pytest.mark.parametrize("kind", ["eye", "classic"])
def test_call_larger_than_the_kept_block(kind):
    """At 1920x1080 the buffers of an eye pass take more than the 2 GiB that a
    context keeps: the call allocates its own and gives them back.  Its rows
    are those of a picture a third as high, whose buffers fit; a pixel's terms
    may be added in another order (80 of one sign: 2 * 80 * 2^-24 < 1e-5)."""
    say("memory: a call larger than the kept block", kind)
    c = P.Context(0)
    ph = P.PhotonSet(c, 5000)
    ph.upload(*random_photons(5000, 1))
    m = P.build_photonmap(c, ph, 1e-3)

    def image(rows):
        sc = P.two_spheres_scene(1920, 360)
        at = sc.camera.screen()  # the first rows keep their rays and random streams
        sc.camera.screen, sc.camera.yreso = lambda: at, rows
        ds = P.DeviceScene(c, sc)
        if kind == "classic":
            return P.trace_classic(c, ds, 3, 1)
        return P.trace_eye(c, ds, m, 3, 1, 0.02 ** 2, max_depth=10)

    small = image(360)
    free = _free()
    large = image(1080)
    assert abs(free - _free()) <= GIB // 64
    assert np.allclose(large[:360], small, rtol=1e-5, atol=0.0) and (large[360:] > 0).any()
    assert np.array_equal(image(360), small)
    c.close()
