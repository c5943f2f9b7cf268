"""Photon gathers by a lane each, shared by a wave, and in the union form give
one estimate: exactly the same with the int64 flux (its sums do not depend on
order), within FP32 summation error (n u, n a few hundred photons) otherwise.
Sizes leave partial groups of 64 pixels; one candidate limit makes every query
shared, one none."""
import numpy as np
import pytest

import hastyrenderer_amd as ha
from hastyrenderer_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("size", [(1, 1), (63, 1), (65, 3), (130, 77)])
def test_gather_forms_agree(size, fixed):
    d = scenes.write_caustic_scene("", width=size[0], height=size[1], n_major=60, n_minor=24, max_depth=8,
                                   as_desc=True)
    sc = ha.Scene.create(**d)
    # about 10,000 photons whatever the film
    frac = 10000.0 / (size[0] * size[1])
    outs = []
    for kw in (dict(gather_share_candidates=1), dict(gather_share_candidates=1 << 30), dict(),
               dict(gather_share_candidates=1, gather_union_factor=50.0)):
        sp = ha.Sppm(sc, 4, initial_radius=0.25, store_fraction=frac, emit_fraction=40.0 * frac,
                     fixed_point_flux=fixed, **kw)
        films = [sp.pass_(k)[0].copy() for k in range(3)]
        i = sp.info()
        outs.append((films, i["gather_queries"], i["gather_candidates"], i["gather_found"], sp.pixels()))
    assert outs[0][3] > 0
    for films, nq, nc, nf, px in outs[1:]:
        assert (nq, nc, nf) == outs[0][1:4]
        assert np.array_equal(px["N"], outs[0][4]["N"])
        for a, b in zip(films, outs[0][0]):
            if fixed:
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
            else:
                np.testing.assert_allclose(a, b, rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("fixed", [True, False])
@pytest.mark.parametrize("limit", [0, 3, 40, 1000])
def test_light_and_heavy_queries_of_one_wave(limit, fixed):
    """Where some of a wave's 64 queries have more candidates than the limit and
    some have not, the wave gathers the light ones and leaves the heavy ones:
    counts are those of every query gathered by its lane, and so is the flux
    (to FP32 summation error, as above)."""
    d = scenes.write_caustic_scene("", width=97, height=61, n_major=60, n_minor=24, max_depth=8, as_desc=True)
    sc = ha.Scene.create(**d)
    outs = []
    for share in (1 << 30, limit):
        sp = ha.Sppm(sc, 4, initial_radius=0.25, store_fraction=2.0, emit_fraction=80.0, fixed_point_flux=fixed,
                     gather_share_candidates=share)
        films = [sp.pass_(k)[0].copy() for k in range(3)]
        i = sp.info()
        outs.append((films, (i["gather_queries"], i["gather_candidates"], i["gather_found"]), sp.pixels()["N"]))
    (ref, counts, n_ref), (got, counts2, n_got) = outs
    assert counts == counts2 and counts[2] > 0
    assert np.array_equal(n_ref, n_got)
    for a, b in zip(ref, got):
        if fixed:
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        else:
            np.testing.assert_allclose(a, b, rtol=1e-4, atol=1e-6)
