"""Rays that are not finite (masked-out entries of a host program's arrays) and
rays from so far out that origin / direction overflows miss in every query form,
and the ordinary rays that share a wave with them keep
their hits.  tests/test_walk_cpu.py walks the same rays on the host with every
index checked."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from test_walk_cpu import nonfinite_rays, overflowing_rays
from test_zz_no_alloc import _Dev, _noalloc

pytestmark = pytest.mark.gpu

RECORD = np.dtype([("geom_id", "<u4"), ("prim_id", "<u4"), ("t", "<f4"), ("u", "<f4"), ("v", "<f4"),
                   ("ng", "<f4", 3)])


def _mixed(every):
    """Ordinary rays with every `every`-th one replaced."""
    bad = np.concatenate([nonfinite_rays(), overflowing_rays()])
    rng = np.random.default_rng(every)
    n = every * len(bad)
    d = rng.normal(size=(n, 3))
    rays = np.concatenate([rng.uniform(-1.2, 2.2, (n, 3)), d / np.linalg.norm(d, axis=1, keepdims=True)],
                          1).astype(np.float32)
    mixed = rays.copy()
    mixed[::every] = bad
    return rays, mixed, np.arange(n) % every == 0


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("every", [1, 2, 7])
def test_unusable_rays_miss(cornell_job, ggx_small_job, every, width):
    rays, mixed, bad = _mixed(every)
    for job in (cornell_job, ggx_small_job):
        sc = ha.Scene(job)
        sc.set_launch_ex(bvh_width=width)
        ref, got = sc.trace_hits(rays), sc.trace_hits(mixed)
        assert (got["geom_id"][bad] == 0xFFFFFFFF).all() and np.isposinf(got["t"][bad]).all()
        assert np.array_equal(got[~bad], ref[~bad])
        _, tri, tuv = sc.trace_closest(mixed)
        assert (tri[bad] == -1).all()
        assert np.array_equal(tri[~bad], sc.trace_closest(rays)[1][~bad])
        n = len(mixed)
        d_rays, d_hits = _Dev(24 * n), _Dev(32 * n)
        d_rays.upload(mixed)
        assert _noalloc(sc, d_rays.ptr, n, d_hits.ptr) == 0
        assert np.array_equal(d_hits.download(32 * n).view(RECORD)["t"], got["t"])
        d_rays.free()
        d_hits.free()
