"""Scenes and tree builds at the limit of a device's HBM budget."""
import numpy as np
import pytest

import xtracer_amd as xa
from tests.helpers import HipBuffers, mixed_rays, scene_path

E_BUDGET = 5


class Rays:
    """Device-resident rays for the trace that allocates nothing."""

    def __init__(self, n, box):
        o, d = mixed_rays(None, n, seed=11, box=box)
        r0, r1 = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
        r0[:, :3], r1[:, :3] = o, d
        r0[:, 3] = np.uint32(xa.HIT_NONE).view(np.float32)
        self.n, self.hip = n, HipBuffers()
        self.r0, self.r1, self.out = self.hip.put(r0), self.hip.put(r1), self.hip.put(np.zeros((n, 4), np.float32))

    def trace(self, dev, sid):
        rc = xa.lib().xt_trace_device_static(dev.handle, sid, xa.ACCEL_KDTREE, self.r0, self.r1, self.out, None, self.n)
        assert rc == 0
        return self.hip.get(self.out, np.zeros((self.n, 4), np.float32)).view(np.uint32)


@pytest.fixture
def rays():
    r = Rays(4096, (-1, 1))
    yield r
    r.hip.free()


def _resident_bytes(scene):
    """Device memory of the scene walked on its kd-tree: what an upload needs at most."""
    i = scene.info()
    per_prim = 48 + 72 + 48 + (36 if i.any_vertex_normals else 0)  # FP32 and FP64 record, texture coordinates, normals
    trees = 48 * i.n_oct_nodes + 4 * i.n_oct_refs + 8 * i.n_kd_nodes + (4 + 48) * i.n_kd_refs
    return per_prim * i.n_prims + trees + (1 << 13)  # planes, materials, objects, rounding of the arrays


@pytest.mark.gpu
@pytest.mark.parametrize("kind,kw", [("strands", {"strands": 600, "step": 0.4}), ("icosphere", {"subdiv": 5}), ("terrain", {"n": 61})])
def test_a_scene_that_fits_is_taken(device, rays, kind, kw):
    """Every budget that holds the scene's arrays, its kd-tree and the copies of
    the leaves takes it, whatever scratch the choice and the build of its index
    could use with more; a released scene's memory is there for the next."""
    scene = xa.Scene(scene_path(kind, **kw))
    sid = device.upload(scene)
    ref = rays.trace(device, sid)
    assert (device.kdtree(sid)[3]["bvh_depth"] == 0) == (kind == "strands")  # both indexes are tried
    device.release(sid)
    assert (ref[:, 1] != xa.HIT_NONE).any()
    need = _resident_bytes(scene)
    for more in (1.0, 1.02, 1.1, 1.25, 1.5, 1.75, 2.0, 2.5, 3.0, 4.0, 6.0):
        dev = xa.Device(0, hbm_budget=int(need * more))
        for _ in range(2):
            sid = dev.upload(scene)
            hit = rays.trace(dev, sid)
            assert np.array_equal(hit[:, 1], ref[:, 1])
            np.testing.assert_allclose(hit[:, 0].view(np.float32), ref[:, 0].view(np.float32), rtol=1e-6)
            dev.release(sid)
        dev.close()
    dev = xa.Device(0, hbm_budget=need // 2)
    with pytest.raises(xa.XtError) as e:
        dev.upload(scene)
    assert e.value.code == E_BUDGET
    dev.close()
def _uploads(scene, budget):
    """Whether a device of this budget takes the scene."""
    dev = xa.Device(0, hbm_budget=budget)
    try:
        dev.upload(scene)
        return True
    except xa.XtError as e:
        assert e.code == E_BUDGET
        return False
    finally:
        dev.close()


def _least_budget(scene, hi, step=1 << 14):
    lo = 0
    assert _uploads(scene, hi)
    while hi - lo > step:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if _uploads(scene, mid) else (mid, hi)
    return hi


@pytest.mark.gpu
def test_refused_rebuild_keeps_the_tree(rays):
    """A rebuild that does not fit the budget leaves the resident tree, its
    leaf copies and its hits as they were; one that fits replaces them."""
    params = dict(kd_leaf_prims=1, kd_cost_intersect=60.0)
    path = scene_path("strands", strands=600, step=0.4)
    scene, finer = xa.Scene(path, threads=1), xa.Scene(path, threads=1, **params)
    assert finer.info().n_kd_refs > scene.info().n_kd_refs
    least = _least_budget(scene, 512 << 20)
    outcomes = []
    for k in range(25):
        dev = xa.Device(0, hbm_budget=int(least * 1.25 ** k))
        sid = dev.upload(scene)
        nodes, refs, bounds, st = dev.kdtree(sid)
        assert st["bvh_depth"] == 0
        hits = rays.trace(dev, sid)
        try:
            dev.build_kd(sid, **params)
            outcomes.append(True)
            want = finer.kdtree()
        except xa.XtError as e:
            assert e.code == E_BUDGET
            outcomes.append(False)
            want = (nodes, refs, bounds)
        got = dev.kdtree(sid)
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert np.array_equal(rays.trace(dev, sid)[:, 1], hits[:, 1])
        # what the failed or finished build held is given back
        dev.release(sid)
        assert np.array_equal(rays.trace(dev, dev.upload(scene)), hits)
        dev.close()
        if outcomes[-3:] == [True] * 3:
            break
    assert not outcomes[0] and outcomes[-1]
    assert outcomes == sorted(outcomes)
