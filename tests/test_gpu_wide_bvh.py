"""The wide BVH and its walk where they can go wrong: soups around the sizes at
which the build changes hands (one leaf, one node, one block's clusters, more),
boxes of no thickness, equal primitives, queues around a wave's first run and
beyond the grid."""
import numpy as np
import pytest

import xtracer_amd as xa
from oracle.oracle import OracleScene
from tests import scn
from tests.helpers import edge_band, plane_point, scene_path, soup_to_object_local


def _soup_scene(tmp_path, tris, spheres=()):
    scn.write_obj(tmp_path / "soup.obj", tris)
    geo = {"soup": dict(type="mesh", source="soup.obj")}
    obj = {"soup": ("soup", "m")}
    for k, (c, r) in enumerate(spheres):
        geo["s%03d" % k] = dict(type="sphere", position=c, radius=r)
        obj["s%03d" % k] = ("s%03d" % k, "m")
    return xa.Scene(scn.write(tmp_path / "scene.scn", geo, obj, {"m": dict(type="lambert", kd=(0.5, 0.5, 0.5))}))


def _rays(n, seed, targets):
    """Rays from a shell around the targets at random points on them, and back."""
    rng = np.random.default_rng(seed)
    o = rng.normal(size=(n, 3))
    o = 9.0 * o / np.linalg.norm(o, axis=1)[:, None]
    aim = targets[rng.integers(len(targets), size=n)] + rng.normal(scale=0.02, size=(n, 3))
    d = aim - o
    d /= np.linalg.norm(d, axis=1)[:, None]
    return o.astype(np.float32), d.astype(np.float32)


def _check(device, s, o, d):
    sid = device.upload(s)
    t, prim, _, _, _ = device.trace(sid, o, d)
    device.release(sid)
    tr, obr, pr, ptr, _ = OracleScene(s).trace(o.astype(np.float64), d.astype(np.float64))
    arr = s.arrays()
    obj, loc = soup_to_object_local(arr, prim)
    same = (obj == obr) & (loc == pr)
    bad = np.flatnonzero(~same)
    # a ray may differ from the oracle only within the edge band of its primitive
    assert edge_band(arr, prim[bad], plane_point(arr, prim[bad], o[bad], d[bad])).all()
    assert same.mean() >= 0.999
    hit = same & (obr >= 0)
    assert hit.any()
    # t is recomputed in 64 bits and rounded once
    np.testing.assert_allclose(t[hit], tr[hit], rtol=1e-5)
    assert np.isinf(t[same & (obr < 0)]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 33, 1023, 1024, 1025, 2500])
def test_soup_sizes(device, tmp_path, n):
    rng = np.random.default_rng(n)
    c = rng.uniform(-2, 2, (n, 1, 3))
    tris = c + rng.normal(scale=0.25, size=(n, 3, 3))
    s = _soup_scene(tmp_path, tris, [((0.0, 0.0, 2.5), 0.5), ((2.5, 0.5, 0.0), 0.25)])
    o, d = _rays(4000, n, np.float32(tris).mean(axis=1))
    _check(device, s, o, d)


@pytest.mark.gpu
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_flat_grid(device, tmp_path, axis):
    """A plane of axis-aligned cells: every box is flat and neighbouring boxes
    share their edges exactly, and so do the rays aimed along the grid lines."""
    k = 24
    g = np.linspace(-1.5, 1.5, k + 1)
    tris = []
    for i in range(k):
        for j in range(k):
            a, b, c, e = [(g[x], g[y]) for x, y in ((i, j), (i + 1, j), (i + 1, j + 1), (i, j + 1))]
            tris += [[a, b, c], [a, c, e]]
    p = np.array(tris)
    p = np.stack([p[..., 0], p[..., 1], np.full(p.shape[:2], 0.375)], axis=-1)
    p = np.roll(p, axis, axis=-1)
    s = _soup_scene(tmp_path, p)
    o, d = _rays(4000, axis, np.float32(p).mean(axis=1))
    # straight down on cell corners, edge middles and cell middles
    h = np.linspace(-1.5, 1.5, 2 * k + 1)[1:-1]
    u, v = np.meshgrid(h, h)
    o2 = np.roll(np.stack([u.ravel(), v.ravel(), np.full(u.size, 5.0)], 1), axis, axis=1)
    d2 = np.roll(np.tile([0.0, 0.0, -1.0], (u.size, 1)), axis, axis=1)
    sid = device.upload(s)
    t, prim, _, _, _ = device.trace(sid, o2.astype(np.float32), d2.astype(np.float32))
    device.release(sid)
    assert (prim != xa.HIT_NONE).all()
    np.testing.assert_allclose(t, 4.625, rtol=1e-6)
    _check(device, s, o, d)


@pytest.mark.gpu
def test_equal_primitives(device, tmp_path):
    """700 copies of one triangle: the tie goes to the first, as in the oracle."""
    tri = np.array([[[-1.0, -1.0, 0.0], [1.0, -1.0, 0.25], [0.0, 1.0, 0.5]]])
    s = _soup_scene(tmp_path, np.repeat(tri, 700, axis=0))
    o, d = _rays(500, 3, np.float32(tri).mean(axis=1))
    _check(device, s, o, d)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 4097, 300007, 1500001])
def test_queue_lengths(device, n):
    """Every ray of a queue is traced, whichever run of whichever wave takes it."""
    s = xa.Scene(scene_path("terrain", n=41))
    sid = device.upload(s)
    o, d = _rays(1009, 5, np.zeros((1, 3)))
    ref = device.trace(sid, o, d)
    k = np.arange(n) % len(o)
    got = device.trace(sid, o[k], d[k])
    device.release(sid)
    assert np.array_equal(got[0].view(np.uint32), ref[0][k].view(np.uint32))
    assert np.array_equal(got[1], ref[1][k])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 3, 64, 1000, 4100, 70000])
def test_lanes_of_a_ray_agree(device, tmp_path, n):
    """Short queues leave lanes to walk parts of other lanes' rays: the hits of
    overlapping, repeated and edge-sharing triangles are those of a queue that
    keeps every lane busy."""
    rng = np.random.default_rng(17)
    c = rng.uniform(-1, 1, (120, 1, 3))
    tris = c + rng.normal(scale=0.9, size=(120, 3, 3))
    fan = np.stack([tris[:, 0], tris[:, 2], tris[:, 2] + (tris[:, 1] - tris[:, 0])], axis=1)  # shares edge 0-2
    s = _soup_scene(tmp_path, np.concatenate([tris, tris, fan, tris[:40]]), [((0.0, 0.0, 0.0), 1.5)])
    edge = 0.5 * (tris[:, 0] + tris[:, 2])
    o, d = _rays(1000, 23, np.float32(np.concatenate([tris.mean(axis=1), edge])))
    sid = device.upload(s)
    k = np.arange(600000) % len(o)
    ref = [a[:1000] for a in device.trace(sid, o[k], d[k])[:2]]
    k = np.arange(n) % len(o)
    got = device.trace(sid, o[k], d[k])
    device.release(sid)
    assert np.array_equal(got[1], ref[1][k])
    assert np.array_equal(got[0].view(np.uint32), ref[0][k].view(np.uint32))
