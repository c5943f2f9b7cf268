"""Ray queries at the edges of their grids: partial waves and blocks, the ray
count at which the grid stops growing, and the overflow slices of both node
widths.  Every ray's hit is the one the CPU oracle finds."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

FULL = 2048 * 256  # rays of one sweep of the largest grid


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("n", [1, 63, 65, 257, FULL - 1, FULL + 3])
def test_hits_at_grid_edges(ggx_small_job, width, n):
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    rays = np.concatenate([rng.uniform(-1.2, 2.2, (n, 3)), d / np.linalg.norm(d, axis=1, keepdims=True)],
                          1).astype(np.float32)
    sc = ha.Scene(ggx_small_job)
    sc.set_launch_ex(bvh_width=width)
    hits = sc.trace_hits(rays)
    gp, tri, tuv = sc.trace_closest(rays)
    assert np.array_equal(hits["geom_id"], gp[:, 0]) and np.array_equal(hits["prim_id"], gp[:, 1])
    assert np.array_equal(hits["t"], tuv[:, 0])
    # the oracle's hits of the first and last rays (the ones at the edges)
    at = np.unique(np.concatenate([np.arange(min(n, 2000)), np.arange(max(0, n - 2000), n)]))
    otri, otuv, _ = po.OracleJob(ggx_small_job).trace(rays[at])
    assert np.array_equal(tri[at], otri)
    assert np.array_equal(tuv[at][otri >= 0], otuv[otri >= 0])
