"""The tree's radius query: one lane per query for counts and lists, four for
sums, whose lanes take a leaf's photons in turn.  Photon counts around the
leaf (32) and the quad's steps, query counts around the blocks, balls of
nothing, some and everything: index sets equal brute force, sums are the
FP64 oracle's within the float bound of the grid's sums, and a query's sum
does not depend on the others in its call."""
import numpy as np
import pytest

import oracle_lib as O
from gpu_common import ctx, random_photons, say
from test_gpu_grid import COS_ABS, RTOL, T_ABS, WMAX

import ppmpa_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_photon", [1, 3, 4, 5, 15, 16, 17, 31, 32, 33, 48, 64, 65, 1025])
@pytest.mark.parametrize("r", [1e-4, 0.11, 2.0])
def test_tree_edges(n_photon, r):
    say("tree edges", n_photon, r)
    c = ctx()
    pos, dir, wl = random_photons(n_photon, 5)
    power = 1.0 / n_photon
    ph = P.PhotonSet(c, n_photon)
    ph.upload(pos, dir, wl)
    m = P.PhotonMap(c, n_photon).build(ph, power)
    om = O.OMap(pos, dir, wl, power)
    rng = np.random.default_rng(6)
    q = rng.uniform(0.0, 1.0, (600, 3))
    q[::5] = pos[rng.integers(0, n_photon, len(q[::5]))]
    nrm = rng.normal(size=q.shape)
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    for refine, mode in ((False, 1), (True, 0)):
        want = O.within_brute(pos, q, r * r, mode=mode)
        for k in (1, 63, 64, 65, 256, 257, 600):
            got = m.within(q[:k], r * r, refine64=refine)
            assert all(np.array_equal(g, w) for g, w in zip(got, want[:k])), (refine, k)
    sets = O.within_brute(pos, q, r * r, mode=1)
    counts = np.array([np.bincount(wl[s], minlength=3) for s in sets], float).reshape(-1, 3)
    qmag = (np.abs(q).max(axis=1) + r) / r
    for pf in (0, 1, 2):
        whole = m.estimate_radiance(q, nrm, r * r, pfilter=pf)
        # the grid's per-entry bound: each photon's cosine and filter weight
        # is off by the rounding of its inputs to float
        want = om.gather(q, nrm, r * r, pf, f32set=True)
        per_term = COS_ABS * WMAX[pf] + (T_ABS * qmag[:, None] if pf else 0.0)
        bound = RTOL * np.abs(want) + power / (np.pi * r * r) * counts * per_term
        assert np.all(whole[want == 0] == 0) and np.all(np.abs(whole - want) <= bound), pf
        for k in (1, 15, 16, 17, 63, 64, 65, 257):
            assert np.array_equal(m.estimate_radiance(q[:k], nrm[:k], r * r, pfilter=pf), whole[:k]), (pf, k)
            assert np.array_equal(m.estimate_radiance(q[-k:], nrm[-k:], r * r, pfilter=pf), whole[-k:]), (pf, k)
