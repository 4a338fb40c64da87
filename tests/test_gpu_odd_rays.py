"""Rays that a walk of the wide BVH could spend itself on: from far away, and
with components that are not finite."""
import numpy as np
import pytest

import xtracer_amd as xa
from tests import scn
from tests.helpers import mixed_rays, scene_path
from xtracer_amd import scenes


@pytest.mark.gpu
@pytest.mark.parametrize("away", [1.0, 30.0, 300.0, 900.0])
def test_no_ray_slips_through_a_closed_mesh(device, tmp_path, away):
    """Rays from `away` extents at a point within 0.9 radii of a sphere's middle:
    FP32 moves its triangles by at most 2.5e-7 * 2 * 900 of their coordinates."""
    v, f = scenes.icosphere(5)
    scn.write_obj(tmp_path / "ball.obj", v[f])
    s = xa.Scene(scn.write(tmp_path / "ball.scn", {"ball": dict(type="mesh", source="ball.obj")},
                           {"ball": ("ball", "m")}, {"m": dict(type="lambert", kd=(0.5, 0.5, 0.5))}))
    rng = np.random.default_rng(int(away))
    u, at = rng.normal(size=(2, 100000, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    at *= (0.9 * rng.random(len(at)) / np.linalg.norm(at, axis=1))[:, None]
    o = (at + 2.0 * away * u).astype(np.float32)
    d = at - o
    d /= np.linalg.norm(d, axis=1)[:, None]
    sid = device.upload(s)
    assert device.kdtree(sid)[3]["bvh_depth"] > 0
    t, prim = device.trace(sid, o, d.astype(np.float32))[:2]
    device.release(sid)
    assert (prim != xa.HIT_NONE).all()
    # the hit lies on the near side of the ball
    p = o + t[:, None].astype(np.float64) * d.astype(np.float32)
    assert (np.abs(np.linalg.norm(p, axis=1) - 1.0) < 0.01 + 1e-6 * away * 2.0).all()
    assert ((p * d).sum(axis=1) < 0).all()


@pytest.mark.gpu
def test_rays_that_are_not_finite_miss(device):
    """Each component of origin or direction NaN or infinite, among ordinary
    rays whose hits stay what they are."""
    s = xa.Scene(scene_path("terrain", n=41))
    sid = device.upload(s)
    assert device.kdtree(sid)[3]["bvh_depth"] > 0
    o, d = mixed_rays(None, 6000, seed=8)
    ref = device.trace(sid, o, d)
    bad = np.arange(3, 6000, 7)
    ob, db = o.copy(), d.copy()
    for k, i in enumerate(bad):
        what = (np.nan, np.inf, -np.inf)[k % 3]
        cols = ([0], [1], [2], [0, 1], [0, 1, 2])[k // 3 % 5]
        (ob if k // 15 % 2 else db)[i, cols] = what
    t, prim, _, _, _ = device.trace(sid, ob, db)
    device.release(sid)
    assert (prim[bad] == xa.HIT_NONE).all() and np.isinf(t[bad]).all()
    good = np.setdiff1d(np.arange(6000), bad)
    assert np.array_equal(prim[good], ref[1][good])
    assert np.array_equal(t[good].view(np.uint32), ref[0][good].view(np.uint32))
