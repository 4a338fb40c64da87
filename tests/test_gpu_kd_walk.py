"""The FP32 walk of the kd-tree, which scenes of long thin slanting triangles
take: every stack size, block size and leaf and node layout against the
oracle, with rays that overflow the shortest ring of pending subtrees."""
import numpy as np
import pytest

import xtracer_amd as xa
from oracle.oracle import OracleScene
from xtracer_amd import scenes
from tests import scn
from tests.helpers import camera_rays, soup_to_object_local
from tests.test_gpu_tuning import DEFAULT, tuned  # noqa: F401

CAM = dict(position=(0.1, 0.05, -3.0), target=(0.0, 0.0, 0.0), fov=30.0)


@pytest.fixture(scope="module")
def hair(tmp_path_factory):
    """16384 needles of any direction across the z axis, one behind the other:
    rays along z leave a far subtree behind at nearly every level of the tree.
    The scene, rays (a camera's, and from anywhere inside, half of them near z)
    and the oracle's hits."""
    rng = np.random.default_rng(5)
    n = 1 << 14
    z = np.linspace(-1, 1, n)
    phi = rng.uniform(0, np.pi, n)
    along = np.stack([np.cos(phi), np.sin(phi), rng.uniform(-0.01, 0.01, n)], 1)
    side = 4e-4 * np.stack([-np.sin(phi), np.cos(phi), np.zeros(n)], 1)
    mid = np.stack([rng.uniform(-0.5, 0.5, n), rng.uniform(-0.5, 0.5, n), z], 1)
    d = tmp_path_factory.mktemp("hair")
    scn.write_obj(d / "hair.obj", np.stack([mid - along - side, mid - along + side, mid + along], 1))
    s = xa.Scene(scn.write(d / "hair.scn", {"hair": dict(type="mesh", source="hair.obj")}, {"hair": ("hair", "m")},
                           {"m": dict(type="lambert", kd=(0.5, 0.5, 0.5))}, camera=CAM))
    o, d = camera_rays(s.camera(), 40, 40)
    o2 = rng.uniform(-0.7, 0.7, (3000, 3))
    d2 = rng.normal(size=(3000, 3)) * np.where(np.arange(3000) % 2, 1.0, 0.05)[:, None] ** np.array([1, 1, 0])
    d2 /= np.linalg.norm(d2, axis=1)[:, None]
    o, d = np.concatenate([o, o2]).astype(np.float32), np.concatenate([d, d2]).astype(np.float32)
    return s, o, d, OracleScene(s).trace(o.astype(np.float64), d.astype(np.float64))


def _pending(nodes, lo, hi, o, d, t_hit):
    """The largest number of far subtrees that a ray has pending on its way to its hit."""
    with np.errstate(divide="ignore", over="ignore", invalid="ignore"):
        a, b = (lo - o) / d, (hi - o) / d
    t0, t1 = max(0.0, np.fmax.reduce(np.fmin(a, b))), np.fmin.reduce(np.fmax(a, b))
    stack, most = ([(0, t0, t1)] if t0 <= t1 else []), 0
    while stack:
        n, t0, t1 = stack.pop()
        if t0 > t_hit:
            break
        while (nodes[n, 0] & 3) != 3:
            axis, child = int(nodes[n, 0] & 3), int(nodes[n, 0] >> 2)
            t = (float(nodes[n, 1:2].view(np.float32)[0]) - o[axis]) / d[axis]
            near, far = (child + 1, child) if d[axis] < 0 else (child, child + 1)
            if t > t1:
                n = near
            elif t < t0:
                n = far
            else:
                stack.append((far, t, t1))
                most = max(most, len(stack))
                n, t1 = near, t
    return most


def test_rays_overflow_the_ring_of_8(hair):
    s, o, d, ref = hair
    nodes, _, b = s.kdtree()
    b = b.astype(float)
    k = np.array([_pending(nodes, b[:3], b[3:], o[i].astype(float), d[i].astype(float), ref[0][i])
                  for i in range(0, len(o), 11)])
    assert (k > 8).mean() > 0.2


def _check(s, got, ref):
    t, prim = got[:2]
    tr, obr, pr = ref[:3]
    obj, loc = soup_to_object_local(s.arrays(), prim)
    same = (obj == obr) & ((obr < 0) | (loc == pr))
    assert same.mean() >= 0.999
    hit = same & (obr >= 0)
    assert hit.mean() > 0.1
    np.testing.assert_allclose(t[hit], tr[hit], rtol=1e-5)
    assert np.isinf(t[same & (obr < 0)]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("stack", [8, 12, 16, 24])
@pytest.mark.parametrize("block", [128, 256])
@pytest.mark.parametrize("per_cu", [1, xa.TUNING_AUTO])
def test_stacks_and_blocks(tuned, hair, stack, block, per_cu):  # noqa: F811
    s, o, d, ref = hair
    sid = tuned.upload(s)
    assert tuned.kdtree(sid)[3]["bvh_depth"] == 0
    tuned.set_tuning(**dict(DEFAULT, kd_stack=stack, trace_block=block, trace_blocks_per_cu=per_cu))
    got = tuned.trace(sid, o, d)
    k = np.arange(300000) % len(o)  # beyond what the grid takes at once with one block a compute unit
    many = tuned.trace(sid, o[k], d[k])
    tuned.release(sid)
    _check(s, got, ref)
    assert np.array_equal(many[1], got[1][k])
    assert np.array_equal(many[0].view(np.uint32), got[0][k].view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("knobs", [{"kd_layout": 2}, {"kd_leaf": 2}, {"trace_segments": 8},
                                   {"kd_layout": 2, "kd_leaf": 2, "trace_segments": 8, "kd_stack": 8, "trace_block": 128}])
def test_layouts(tuned, hair, knobs):  # noqa: F811
    s, o, d, ref = hair
    tuned.set_tuning(**dict(DEFAULT, **knobs))
    sid = tuned.upload(s)  # kd_layout applies to scenes uploaded afterwards
    _check(s, tuned.trace(sid, o, d), ref)
    # the octree's walk tests the same triangles with the same arithmetic; the
    # oracle's image may differ where a ray passes a needle's edge within what
    # FP32 places it (1e-3 of its width)
    W, H, spp = 72, 56, 2
    job = dict(integrator=xa.DEPTH, width=W, height=H, camera=s.camera(), samples=spp, seed=4)
    img, st = tuned.render(xa.make_job(sid, **job))
    octree, st2 = tuned.render(xa.make_job(sid, accel=xa.ACCEL_OCTREE, **job))
    tuned.release(sid)
    assert np.array_equal(img.view(np.uint32), octree.view(np.uint32)) and st.queries == st2.queries
    want, nq = OracleScene(s).render(xa.DEPTH, W, H, scenes.camera_dict(**CAM), samples=spp, seed=4)
    assert st.queries == nq
    assert (img == want).all(axis=2).mean() >= 0.999


@pytest.mark.gpu
def test_device_built_tree(tuned, hair):  # noqa: F811
    """The walk on trees that the device built, with default and other parameters."""
    s, o, d, ref = hair
    tuned.set_tuning(**DEFAULT)
    sid = tuned.upload(s)
    for params in (dict(), dict(kd_leaf_prims=2), dict(kd_max_depth=9), dict(kd_cost_intersect=40.0)):
        assert tuned.build_kd(sid, **params)["bvh_depth"] == 0
        _check(s, tuned.trace(sid, o, d), ref)
    tuned.release(sid)
