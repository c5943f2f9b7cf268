"""The path pool's record packing and results ring at the sizes where they can
go wrong: pools of one record, of a partial wave and of a partial block, jobs
with and without late light samples and media texels in one batch, and a
render longer than the results ring.  Images never depend on any of it."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from hastyrenderer_amd import scenes

pytestmark = pytest.mark.gpu


def _render(scene, seed, first, n):
    info = scene.info()
    f = ha.DeviceFilms(info["width"], info["height"])
    scene.render_pt_device(seed, first, n, *f.ptrs)
    out = f.download()
    f.close()
    return out


def _same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("slots", [1, 63, 64, 65, 257, 1023])
def test_pool_size_changes_nothing(cornell_job, slots):
    sc = ha.Scene(cornell_job)
    sc.set_settings(width=19, height=7)
    ref = _render(sc, 4, 0, 5)
    sc.set_launch(path_slots=slots)
    _same(ref, _render(sc, 4, 0, 5))


@pytest.mark.parametrize("slots", [100, 1 << 16])
def test_batch_of_unlike_jobs(tmp_path, cornell_job, slots):
    """Late light samples (sky and light), media texels and plain jobs share
    one pool."""
    jobs = [scenes.write_cornell(str(tmp_path / "sky"), width=33, height=21, sky=True),
            scenes.write_textured_scene(str(tmp_path / "tex"), width=40, height=23), cornell_job]
    scs = [ha.Scene(j) for j in jobs]
    scs[2].set_settings(width=50, height=31)
    alone = [_render(sc, 7 + k, 0, 3) for k, sc in enumerate(scs)]
    films = [ha.DeviceFilms(sc.info()["width"], sc.info()["height"]) for sc in scs]
    scs[0].set_launch(path_slots=slots)
    ha.render_batch([(sc, 7 + k, 0, 3, f) for k, (sc, f) in enumerate(zip(scs, films))])
    for f, ref in zip(films, alone):
        _same(f.download(), ref)


@pytest.mark.parametrize("which", ["cornell", "ggx_small", "caustic_small"])
@pytest.mark.parametrize("size", [(5, 3), (97, 41), (701, 402)])
def test_finished_paths_equal_bounce_by_bounce(which, size, request):
    """The last 2^18 paths of a render run to their ends one by one; a render
    by captured graphs runs every bounce of every path through the bounce
    kernels.  15 paths, a partial grid, and more than 2^18."""
    sc = ha.Scene(request.getfixturevalue(which + "_job"))
    sc.set_settings(width=size[0], height=size[1])
    sc.set_launch_ex(use_graph=1)
    ref = _render(sc, 9, 0, 1)
    sc.set_launch_ex(use_graph=0)
    _same(ref, _render(sc, 9, 0, 1))


def test_render_longer_than_the_ring(cornell_job):
    """36 samples of a 2048 x 2048 film are more than the ring's 2^27 paths."""
    sc = ha.Scene(cornell_job)
    sc.set_settings(width=2048, height=2048, max_depth=3)
    f = ha.DeviceFilms(2048, 2048)
    sc.render_pt_device(1, 0, 36, *f.ptrs)
    whole = f.download()
    f.zero()
    for first, n in ((0, 7), (7, 28), (35, 1)):
        sc.render_pt_device(1, first, n, *f.ptrs)
    _same(whole, f.download())
    f.close()
