"""The shade takes queries in groups of 64 from a grid sized for a full GPU;
waves past one per group leave at once, and each step's records are loaded
while the last ones are tested.  Query counts around the group and block
edges, radii from none to all photons in every ball, and photon counts around
the four-record steps: each result equals, bit for bit, that of the same
query in a call of its own size class (the whole set at once), and the index
sets equal brute force."""
import numpy as np
import pytest

from gpu_common import ctx, random_photons, say

import ppmpa_amd as P

pytestmark = pytest.mark.gpu

N = 1500


@pytest.mark.parametrize("n_photon", [1, 3, 4, 5, 257, 4000])
@pytest.mark.parametrize("r", [1e-4, 0.07, 2.0])
def test_query_counts(n_photon, r):
    say("shade groups", n_photon, r)
    c = ctx()
    pos, dir, wl = random_photons(n_photon, 3)
    ph = P.PhotonSet(c, n_photon)
    ph.upload(pos, dir, wl)
    m = P.PhotonMap(c, n_photon).build_grid(ph, 1.0, r * r)
    rng = np.random.default_rng(4)
    q = rng.uniform(0.0, 1.0, (N, 3))
    q[::7] = pos[rng.integers(0, n_photon, len(q[::7]))]
    nrm = rng.normal(size=(N, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    whole = m.estimate_radiance(q, nrm, r * r)
    for k in (1, 63, 64, 65, 128, 255, 256, 257, 513, 1023):
        assert np.array_equal(m.estimate_radiance(q[:k], nrm[:k], r * r), whole[:k]), k
        assert np.array_equal(m.estimate_radiance(q[-k:], nrm[-k:], r * r), whole[-k:]), k
    f, p = q[:200].astype(np.float32), pos.astype(np.float32)
    d = f[:, None, :] - p[None, :, :]
    d2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
    for i, got in enumerate(m.within(q[:200], r * r)):
        assert np.array_equal(got, np.nonzero(d2[i] <= np.float32(r * r))[0])
