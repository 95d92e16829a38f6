"""Arrays that cross to and from the device in slots of staging memory (1 MiB
less 256 bytes, eight of them): one slot, a slot more or less than full, several
(copied by several threads), and more than the ring holds."""
import numpy as np
import pytest

from gpu_common import ctx, say

import ppmpa_amd as P

pytestmark = pytest.mark.gpu

SLOT = (1 << 20) - 256
PHOTONS = SLOT // 53  # photons per slot: six doubles, a word and a byte each


def _photons(n, seed=1):
    rng = np.random.default_rng(seed)
    d = rng.standard_normal((n, 3))
    return rng.random((n, 3)), d / np.linalg.norm(d, axis=1, keepdims=True), rng.integers(0, 3, n).astype(np.uint8)


@pytest.mark.parametrize("n", [1, PHOTONS - 1, PHOTONS, PHOTONS + 1, 3 * PHOTONS, 4 * PHOTONS, 9 * PHOTONS + 5,
                               21 * PHOTONS - 1])
def test_photons_come_back(n):
    say("staging photons", n)
    pos, d, wl = _photons(n)
    ph = P.PhotonSet(ctx(), n)
    ph.upload(pos, d, wl)
    gpos, gdir, gwl, meta = ph.download()
    assert np.array_equal(gpos, pos.astype(np.float32).astype(np.float64))
    # the upload normalises in double before it rounds
    assert np.abs(gdir - d).max() <= 2.0 ** -23
    assert np.array_equal(gwl, wl) and np.array_equal(meta & 3, wl)
    assert np.array_equal(meta >> 7, np.arange(n))


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("per", [24, 32, 56])  # bytes per item of the slots: results, queries
def test_gather_the_same_in_pieces(per, refine):
    """Values of many queries at once equal those of the same queries in calls
    that fill no slot; a query that is refused in the last slot leaves the next
    call as it was."""
    say("staging gather", per, refine)
    c = ctx()
    pos, d, wl = _photons(20000, 2)
    ph = P.PhotonSet(c, 20000)
    ph.upload(pos, d, wl)
    m = P.build_photonmap(c, ph, 1e-3)
    for n in (SLOT // per - 1, SLOT // per, SLOT // per + 1, 9 * (SLOT // per) + 3):
        q, nrm, _ = _photons(n, 3)
        full = m.estimate_radiance(q, nrm, 0.03 ** 2, refine64=refine)
        step = 9001
        parts = [m.estimate_radiance(q[i:i + step], nrm[i:i + step], 0.03 ** 2, refine64=refine)
                 for i in range(0, n, step)]
        assert full.any() and np.array_equal(full, np.concatenate(parts))
        bad = q.copy()
        bad[-1, 1] = np.inf
        with pytest.raises(Exception):
            m.estimate_radiance(bad, nrm, 0.03 ** 2, refine64=refine)
        assert np.array_equal(m.estimate_radiance(q[-10:], nrm[-10:], 0.03 ** 2, refine64=refine), full[-10:])
