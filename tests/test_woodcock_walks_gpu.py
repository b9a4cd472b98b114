"""Woodcock walks in rounds and in groups of lanes against the plain walk. The counting kernels walk
one collision at a time, the others up to four a round and the last 16 (then 4) walks of a wave in
groups of lanes; every decision and draw is the same, so frames, estimates and seeds must agree bit
for bit, on films that leave 1 to 64 walks in a wave, for media from nearly empty (walks of
crossings) to a majorant far above the sampled values (walks of hundreds of rejected collisions),
with and without clipping objects. The oracle checks the plain walk's decisions."""
import numpy as np
import pytest

import exposure_render as er
import oracle as O
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _scene(w, h, density, spike, clip):
    sc = scenes.config_ct(scale=0.16, bilateral=False)
    sc.tracer.settings.sampler = capi.SAMPLER_WOODCOCK
    sc.tracer.settings.density_scale = density
    sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = w, h
    if spike:      # one voxel in eight along each axis raises its macrocell's majorant
        sc.voxels[4::8, 4::8, 4::8] = 4095
    if clip:
        tm, inv = scenes.look_at((0.2, 0.1, 0.3), (1.0, 0.5, 0.2))
        sc.add_clip(scenes.clipping_shape(capi.SHAPE_BOX, tm, inv, size=(0.5, 0.6, 0.4)))
    return sc


@pytest.mark.parametrize("clip", [False, True])
@pytest.mark.parametrize("density,spike", [(0.5, True), (30.0, True), (300.0, True), (100.0, False)])
@pytest.mark.parametrize("w,h", [(1, 1), (2, 2), (5, 3), (9, 8), (131, 70)])
def test_walks_agree(fresh, w, h, density, spike, clip):
    sc = _scene(w, h, density, spike, clip)
    seeds = O.seeds_for(w, h, 31)
    got = []
    for counting in (False, True):
        print(f"[walks] {w}x{h} density {density} spike {spike} clip {clip} counting {counting}", flush=True)
        r = er.Renderer(sc)
        r.set_seeds(*seeds)
        r.set_counting(counting)
        r.render_passes(4)
        got.append((r.frame(), r.running(), r.get_seeds()))
        r.close()
    a, b = got
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    assert np.array_equal(a[2][0], b[2][0]) and np.array_equal(a[2][1], b[2][1])
    orc = O.Oracle(sc)
    orc.compute_gm_max()
    s1, s2 = seeds[0].copy(), seeds[1].copy()
    for _ in range(4):
        frame = orc.trace(s1, s2)[0]
    assert np.array_equal(a[2][0], s1) and np.array_equal(a[2][1], s2)
    assert np.array_equal(a[0][..., 3], frame[..., 3])
