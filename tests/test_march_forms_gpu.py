"""The marches' specialised forms against their general one. Which form a pass takes follows from the
scene (clipping objects, sampler, sign of the opacity) and from whether samples are counted: the
counting kernels always take the general form, so a pass with counting on and one with counting
off must agree bit for bit, whatever the launch configuration; the oracle checks the scene itself."""
import numpy as np
import pytest

import exposure_render as er
import oracle as O
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _negative(sc):
    """opacity below zero in a band: the optical depth falls there"""
    t = sc.tracer
    t.opacity.init()
    t.opacity.add(0.0, 0.0).add(300.0, 0.0).add(900.0, -0.05).add(1500.0, 0.3).add(4095.0, 1.0)


def _wide(sc):
    """values up to 65535: the opacity table stays in global memory"""
    sc.voxels[:] = np.minimum(sc.voxels.astype(np.uint32) * 16, 65535).astype(np.uint16)
    t = sc.tracer
    t.opacity.init()
    t.opacity.add(0.0, 0.0).add(4800.0, 0.0).add(24000.0, 0.3).add(65535.0, 1.0)


def _clips(sc):
    tm, inv = scenes.look_at((0.2, 0.1, 0.3), (1.0, 0.5, 0.2))
    sc.add_clip(scenes.clipping_shape(capi.SHAPE_BOX, tm, inv, size=(0.5, 0.6, 0.4)))
    tm, inv = scenes.translate((-0.1, 0.0, 0.1))
    sc.add_clip(scenes.clipping_shape(capi.SHAPE_SPHERE, tm, inv, outer=0.45, invert=1))


def _lens(sc):
    sc.tracer.camera.aperture_size, sc.tracer.camera.focal_distance = 0.02, 2.0


def _dense(sc):
    sc.tracer.settings.density_scale = 2000.0      # most rays end at their first samples


def _thin(sc):
    sc.tracer.settings.density_scale = 3.0         # most rays cross the volume


SCENES = {
    "full": ({}, None), "compat": ({"estimator": capi.ESTIMATOR_COMPAT}, _lens), "negative": ({}, _negative),
    "wide": ({}, _wide), "clips": ({}, _clips), "clips_wide": ({}, lambda sc: (_clips(sc), _wide(sc))),
    "clips_negative": ({}, lambda sc: (_clips(sc), _negative(sc))), "dense": ({}, _dense), "thin": ({}, _thin),
    "woodcock": ({}, lambda sc: setattr(sc.tracer.settings, "sampler", capi.SAMPLER_WOODCOCK)),
    "woodcock_clips": ({}, lambda sc: (_clips(sc), setattr(sc.tracer.settings, "sampler", capi.SAMPLER_WOODCOCK))),
}
#: rays per wave, shadow rays per wave, heavy tiles, heavy rays per wave, brick
TUNES = [(64, 64, 0, 4, 8), (16, 16, 0, 4, 4), (4, 4, 0, 4, 8), (1, 64, 0, 4, 8), (64, 16, 64, 16, 4), (64, 64, 64, 4, 8),
         (64, 64, 64, 1, 2)]


def _scene(kind):
    kw, edit = SCENES[kind]
    sc = scenes.config_ct(scale=0.16, bilateral=False, **kw)
    sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = 133, 75
    if edit:
        edit(sc)
    return sc


@pytest.mark.parametrize("kind", sorted(SCENES))
def test_forms_agree(fresh, kind):
    sc = _scene(kind)
    orc = O.Oracle(sc)
    if sc.tracer.settings.estimator == capi.ESTIMATOR_FULL:
        orc.compute_gm_max()
    seeds = O.seeds_for(133, 75, 9)
    s1, s2 = seeds[0].copy(), seeds[1].copy()
    frames = [orc.trace(s1, s2)[0] for _ in range(3)]
    for rpw, srpw, heavy, hrpw, brick in TUNES:
        if kind.endswith("wide") and brick == 2:
            continue
        got = []
        for counting in (False, True):
            print(f"[forms] {kind} rays per wave {rpw}/{srpw} heavy {heavy}x{hrpw} brick {brick} counting {counting}", flush=True)
            r = er.Renderer(sc)
            r.set_tune(brick, 8, 7, 4, heavy, rpw, srpw, hrpw)
            r.set_seeds(*seeds)
            r.set_counting(counting)
            r.render_passes(3)
            got.append((r.frame(), r.running(), r.get_seeds()))
            r.close()
        a, b = got
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
        assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
        if "negative" in kind:
            continue      # a macrocell without positive opacity counts as empty, which the oracle does not know
        assert np.array_equal(a[2][0], s1) and np.array_equal(a[2][1], s2)
        assert np.array_equal(a[0][..., 3], frames[2][..., 3])
        np.testing.assert_allclose(a[0], frames[2], rtol=1e-4, atol=1e-6)
