"""One-job renders whose passes are large enough for two pixel groups by default."""
import numpy as np
import pytest

import xtracer_amd as xa
from tests.helpers import scene_path
from tests.test_gpu_tuning import DEFAULT, tuned  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("integrator", [xa.PATHTRACER, xa.AO, xa.NORMAL, xa.DEPTH])
@pytest.mark.parametrize("ray_order", [1, 2, 3])
def test_two_groups_same_bits(tuned, integrator, ray_order):  # noqa: F811
    """Two passes of 552,000 paths each (8625 tiles of 8x8, an odd number), in
    one group and in two: the same bits and queries, also where all paths end
    long before the depth limit of 100 (the early stop)."""
    s = xa.Scene(scene_path("spheres"))
    sid = tuned.upload(s)
    W, H, spp = 1000, 552, 2
    job = xa.make_job(sid, integrator, W, H, s.camera(), samples=spp, rdepth=100, seed=21)
    tuned.set_tuning(**dict(DEFAULT, wave_paths=W * H, ray_order=ray_order, frame_lanes=1))
    ref, one = tuned.render(job)
    tuned.set_tuning(frame_lanes=2)
    img, two = tuned.render(job)
    tuned.release(sid)
    assert one.passes == two.passes == 2
    assert two.trace_launches > one.trace_launches  # two groups were formed
    if integrator == xa.PATHTRACER:
        assert one.trace_launches < 2 * 100  # and stopped early
    assert two.queries == one.queries
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("kind,kw,groups", [("terrain", {"n": 41}, 2), ("spheres", {}, 1)])
def test_octree_frames_in_two_groups(tuned, kind, kw, groups):  # noqa: F811
    s = xa.Scene(scene_path(kind, **kw))
    sid = tuned.upload(s)
    job = xa.make_job(sid, xa.PATHTRACER, 72, 56, s.camera(), samples=3, rdepth=6, seed=4, accel=xa.ACCEL_OCTREE)
    tuned.set_tuning(**dict(DEFAULT, frame_lanes=1))
    ref, one = tuned.render(job)
    tuned.set_tuning(frame_lanes=2)
    img, two = tuned.render(job)
    tuned.release(sid)
    # the early stop may end one group's rounds before the other's
    assert (two.trace_launches > one.trace_launches) == (groups == 2)
    assert two.queries == one.queries
    assert np.array_equal(img.view(np.uint32), ref.view(np.uint32))
