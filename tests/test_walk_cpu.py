"""The BVH walk on the host (tests/csrc/walk_host.hip: the renderer's own slab
test, leaf step and triangle test, every index checked): rays that are not
finite and rays whose slab arithmetic overflows stay inside the tree and miss,
and every other ray's hit is the one the triangle test finds over all
triangles.  Trees with empty slots, both node widths."""
import ctypes as C
import itertools

import numpy as np
import pytest

from conftest import load_testkernels

INF, NAN = np.inf, np.nan


def _walk(tris, width, rays):
    L = load_testkernels()
    rays = np.ascontiguousarray(rays, np.float32)
    tris = np.ascontiguousarray(tris, np.float32).reshape(-1, 9)
    n = len(rays)
    tri, status, tuv = np.empty(n, np.int32), np.empty(n, np.int32), np.empty((n, 3), np.float32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    assert L.tk_walk_host(p(tris), C.c_uint32(len(tris)), C.c_int(width), p(rays), C.c_uint32(n), p(tri), p(tuv),
                          p(status)) == 0
    return tri, tuv, status


def _soup(n, seed=3):
    """n small triangles in [-1, 1]^3."""
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(size=(n, 3, 3)) * 0.15).astype(np.float32)


def _rays(n, seed=5):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    return np.concatenate([rng.uniform(-1.5, 1.5, (n, 3)), d / np.linalg.norm(d, axis=1, keepdims=True)], 1)


def nonfinite_rays():
    """Every mix of an ordinary value, NaN and both infinities in the origin
    or in the direction (the other one ordinary, or not finite throughout)."""
    values = (0.3, NAN, INF, -INF)
    mixes = [m for m in itertools.product(values, repeat=3) if not np.isfinite(m).all()]
    rays = []
    for m in mixes:
        rays += [m + (0.5, -0.6, 0.7), (0.1, 0.2, -0.3) + m]
    for a, b in itertools.product((NAN, INF, -INF), repeat=2):
        rays.append((a,) * 3 + (b,) * 3)
    return np.array(rays, np.float32)


def overflowing_rays():
    """Finite rays for which origin / direction exceeds the largest float."""
    return np.array([(s * b,) * 3 + (x, y, z) for b in (1e19, 1e30, 3e38) for s in (-1.0, 1.0)
                     for x, y, z in itertools.product((0.0, -0.0, 1e-20, -1e-20, 1e-38, 1.0, 3e38), repeat=3)],
                    np.float32)


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("ntris", [0, 1, 2, 5, 21, 300])
def test_nonfinite_rays_miss(ntris, width):
    tri, tuv, status = _walk(_soup(ntris), width, nonfinite_rays())
    assert (status == 0).all()
    assert (tri == -1).all() and np.isposinf(tuv[:, 0]).all()


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("ntris", [1, 2, 5, 21])
def test_overflowing_slabs_stay_in_the_tree(ntris, width):
    rays = overflowing_rays()
    tris = _soup(ntris)
    tri, _, status = _walk(tris, width, rays)
    assert (status == 0).all()
    assert np.array_equal(tri, _walk(tris, 0, rays)[0])


@pytest.mark.parametrize("width", [4, 8])
@pytest.mark.parametrize("ntris", [1, 2, 5, 21, 300])
@pytest.mark.parametrize("offset", [0.0, 1e5, 1e20])
def test_finite_rays_hit_what_the_triangle_test_finds(ntris, width, offset):
    """Scattered and axis-parallel rays, also where the scene lies so far out
    along x that an axis-parallel ray's origin / direction overflows."""
    tris = _soup(ntris)
    rays = _rays(3000)
    rays[::3, 3:] = np.eye(3)[np.arange(1000) % 3] * np.where(np.arange(1000) % 2, 1.0, -1.0)[:, None]
    if offset == 1e20:  # slabs in x: the spacing of floats at 1e20 is 8.8e12
        tris[:, :, 0] *= 1e14
        rays[:, 0] *= 1e14
        rays[:, 3:] = [0.0, 0.0, 1.0]
    tris[:, :, 0] += np.float32(offset)
    rays = rays.astype(np.float32)
    rays[:, 0] += np.float32(offset)
    tri, tuv, status = _walk(tris, width, rays)
    btri, btuv, _ = _walk(tris, 0, rays)
    assert (status == 0).all()
    assert np.array_equal(tri, btri) and np.array_equal(tuv, btuv)
    assert ntris < 300 or (btri >= 0).sum() > 100
