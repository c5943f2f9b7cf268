"""Box tests must not cull what the exact ray enters, wherever the ray starts:
origins inside the scene, at its faces, and up to 1e6 scene sizes away (on
both sides of the distance at which the fused slab test's error bound turns
from a widened box into a relative one), axis-parallel and nearly axis-parallel
directions.  Every hit equals the oracle's watertight test over all triangles
(no BVH)."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _rays(n, scale, rng, axis_eps):
    target = rng.uniform(-1.0, 1.0, (n, 3)) + [0.0, 1.0, 0.0]
    d = rng.normal(size=(n, 3))
    if axis_eps is not None:  # one dominant axis, the others zero or tiny
        k = rng.integers(0, 3, n)
        d = rng.normal(size=(n, 3)) * axis_eps
        d[np.arange(n), k] = rng.choice([-1.0, 1.0], n)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = target - d * scale * rng.uniform(0.1, 1.0, (n, 1))
    return np.concatenate([o, d], 1).astype(np.float32)


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("axis_eps", [None, 0.0, 1e-12, 1e-4])
@pytest.mark.parametrize("scale", [0.5, 3.0, 6.0, 50.0, 1e3, 1e6])
def test_far_and_axis_parallel_rays(cornell_job, ggx_small_job, scale, axis_eps, width):
    rng = np.random.default_rng(int(scale * 10) + width)
    rays = _rays(1500, scale, rng, axis_eps)
    hit_any = False
    for job in (cornell_job, ggx_small_job):
        sc = ha.Scene(job)
        sc.set_launch_ex(bvh_width=width)
        _, tri, tuv = sc.trace_closest(rays)
        otri, otuv, _ = po.OracleJob(job).trace(rays, brute=True)
        assert np.array_equal(tri, otri)
        hit = otri >= 0
        assert np.array_equal(tuv[hit], otuv[hit])
        hit_any = hit_any or hit.any()
    assert hit_any
