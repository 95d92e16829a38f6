"""The eye waves take tiles in fewer parts beyond 8192 tiles: a scene whose
paths branch whole instead of in halves, one of more than 512 shapes in halves
instead of in quarters.  Beside that line a picture's rows are those of the
picture that has one more row of tiles, and both are the oracle's."""
import numpy as np
import pytest

from gpu_common import check_eye_crn, ctx, say, small_scene

import ppmpa_amd as P

pytestmark = pytest.mark.gpu

WIDTH, ROWS, MORE = 1024, 512, 520  # 8192 tiles, and a row of them more


def _scene(kind, rows):
    sc = P.mesh_scene(WIDTH, ROWS, subdiv=3, n_spheres=12, seed=4) if kind == "mesh" else small_scene(kind, WIDTH, ROWS)
    at = sc.camera.screen()  # the first rows keep their rays and random streams
    sc.camera.screen, sc.camera.yreso = lambda: at, rows
    return sc


@pytest.mark.parametrize("kind", ["caustic", "two_spheres", "mesh"])
def test_rows_the_same_on_both_sides(kind):
    """A pixel's terms are the same on both sides and only added in another
    order; 80 terms of one sign each way: 2 * 80 * 2^-24 < 1e-5."""
    say("eye line rows", kind)
    c = ctx()
    img = []
    for rows in (ROWS, MORE):
        s = P.Session(c, P.DeviceScene(c, _scene(kind, rows)),
                      P.pass_cfg(seed=2, n_photon=20000, radius0=0.03, alpha=2.0 / 3.0, max_depth=8))
        s.run(1)
        img.append(s.image(False)[0])
        s.close()
    a, b = img[0], img[1][:ROWS]
    assert a.mean() > 0 and (img[1][ROWS:] > 0).any()
    assert np.allclose(a, b, rtol=1e-5, atol=0.0), np.abs(a - b).max()


@pytest.mark.parametrize("rows", [ROWS, MORE])
def test_caustic_matches_oracle(rows):
    say("eye line oracle caustic", rows)
    check_eye_crn(ctx(), _scene("caustic", rows), 5, 40000, 0.02 ** 2, True, 16)


@pytest.mark.parametrize("rows", [ROWS, MORE])
def test_mesh_matches_oracle(rows):
    """Without direct light (25 shadow rays a query over 1298 shapes, one by
    one in the oracle); the scene's mirrors and glass as in the other meshes'
    comparisons."""
    say("eye line oracle mesh", rows)
    check_eye_crn(ctx(), _scene("mesh", rows), 5, 20000, 0.03 ** 2, False, 8, frac_min=0.97)
