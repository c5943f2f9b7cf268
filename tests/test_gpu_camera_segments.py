"""Photon-mapping camera paths in segments of vertices: paths that end before,
at and after the vertices where they are packed anew, media stacks and
wavelengths carried over them, films of one pixel and of partial blocks.  The
films equal the oracle's."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from conftest import rel_ok
from hastyrenderer_amd import scenes
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [0, 1, 2, 3, 4, 7, 8, 16])
@pytest.mark.parametrize("size", [(1, 1), (67, 41)])
def test_segments_against_the_oracle(tmp_path, depth, size):
    w, h = size
    job = scenes.write_caustic_scene(str(tmp_path), width=w, height=h, n_major=60, n_minor=24, max_depth=depth)
    sc = ha.Scene(job)
    sp = ha.Sppm(sc, 3)
    o = po.OracleSppm(job, seed=3)
    for k in range(2):
        color, normal, albedo = sp.pass_(k)
        ref = o.run_pass(k, w, h)
        assert rel_ok(color, ref[0]).mean() >= 0.999
        assert np.array_equal(normal, ref[1]) and np.array_equal(albedo, ref[2])
