"""The eye waves take a tile of 64 pixels whole, in halves or in quarters, by
the scene and the number of tiles.  Whatever the split, a pixel's image is the
oracle's: odd image sizes (tiles over the edge), every tile shape, with and
without branching paths, beside the rule's lines."""
import numpy as np
import pytest

from gpu_common import ctx, say, small_scene

import oracle_lib as O
import ppmpa_amd as P

pytestmark = pytest.mark.gpu


def _scene(kind, w, h):
    if kind == "mesh":
        return P.mesh_scene(w, h, subdiv=3, n_spheres=12, seed=4)
    return small_scene(kind, w, h)


@pytest.mark.parametrize("kind", ["caustic", "two_spheres", "mesh"])
@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (61, 33)])
@pytest.mark.parametrize("width", [4, 8, 32])
def test_pass_matches_oracle(kind, w, h, width):
    say("eye parts", kind, w, h, width)
    sc = _scene(kind, w, h)
    cfg = P.pass_cfg(seed=2, n_photon=4000, radius0=0.05, alpha=2.0 / 3.0, max_depth=8)
    c = ctx()
    s = P.Session(c, P.DeviceScene(c, sc), cfg)
    s.set_tile_width(width)
    s.run(1)
    mean = s.image(False)[0]
    s.close()
    omean = O.OScene(sc).run_passes(cfg, 1)[0]
    close = (np.abs(mean - omean) <= 1e-3 * np.maximum(np.abs(omean), 1e-3 * np.abs(omean).max())).all(axis=2)
    assert close.mean() > 0.95


@pytest.mark.parametrize("w,h", [(1024, 512), (1024, 520)])  # 8192 tiles, and a row more
def test_images_reproducible_at_the_line(w, h):
    """Two sessions give the same bits (but for overflowed pixels), and the
    image beside the line differs from its neighbour's only by its rows."""
    say("eye parts line", w, h)
    c = ctx()
    ds = P.DeviceScene(c, small_scene("caustic", w, h))
    img = []
    for _ in range(2):
        s = P.Session(c, ds, P.pass_cfg(seed=2, n_photon=4000, radius0=0.05, alpha=2.0 / 3.0, max_depth=8))
        s.run(2)
        img.append(s.image(False)[0])
        s.close()
    assert np.allclose(img[0], img[1], rtol=1e-6, atol=0.0) and (img[0] == img[1]).mean() >= 0.99
    assert img[0].mean() > 0
