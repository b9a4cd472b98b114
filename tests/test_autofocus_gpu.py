"""GetAutoFocusDistance on the GPU: one wave per ray, each ray's place in the draw stream found
from the box tests of the rays before it. The oracle takes the same rays one after the other on
one stream, so the distances are equal bit for bit - also where some or all rays miss the box,
where the places move, and where the rays start inside it."""
import numpy as np
import pytest

import exposure_render as er
import oracle as O
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _scene(kind):
    estimator = capi.ESTIMATOR_COMPAT if kind == "compat" else capi.ESTIMATOR_FULL
    sc = scenes.config_small(scale=0.5, estimator=estimator)
    if kind == "clipped":
        sc.add_clip(scenes.clipping_box((0.25, 0.0, 0.0), (0.5, 1.1, 1.1)))
    if kind == "wide_values":          # an opacity table too large for LDS
        sc.voxels[:] = np.minimum(sc.voxels.astype(np.uint32) * 8, 65535).astype(np.uint16)
        sc.tracer.opacity.init()
        sc.tracer.opacity.add(0.0, 0.0).add(3200.0, 0.0).add(12000.0, 0.6).add(65535.0, 1.0)
    if kind == "inside":
        scenes.set_camera(sc.tracer, sc.film, (0.1, 0.05, 0.2), (0.0, 0.0, 0.0), exposure=4.0)
    if kind == "woodcock":
        sc.tracer.settings.sampler = capi.SAMPLER_WOODCOCK
    return sc


@pytest.mark.parametrize("kind", ["full", "compat", "clipped", "wide_values", "inside", "woodcock"])
def test_autofocus_matches_the_sequential_rays(fresh, kind):
    sc = _scene(kind)
    r = er.Renderer(sc)
    orc = O.Oracle(sc)
    W, H = sc.film
    # the centre, a column across the volume's outline (some rays miss its box), a corner (all miss)
    points = [(W // 2, H // 2)] + [(x, H // 2) for x in range(0, W // 2, 3)] + [(0, 0), (W - 1, H - 1)]
    for u, v in points:
        d = r.autofocus_distance(u, v)
        ref = orc.autofocus(u, v, *r.autofocus_seeds(u, v))
        assert d == ref, (kind, u, v, d, ref)
        assert r.autofocus_distance(u, v) == d
    r.close()


def test_first_call_of_a_tracer(fresh):
    """The call that makes a tracer's workspace, in memory that earlier tracers gave back: its
    arrival count has to be cleared before the kernel counts in it."""
    sc = _scene("full")
    orc = O.Oracle(sc)
    W, H = sc.film
    for k in range(12):
        r = er.Renderer(sc)
        if k % 2:
            r.render_passes(2)      # tables already built, nothing else waits for the device
        d = r.autofocus_distance(W // 2 + k, H // 2)
        assert d == orc.autofocus(W // 2 + k, H // 2, *r.autofocus_seeds(W // 2 + k, H // 2)), k
        assert r.autofocus_distance(W // 2 + k, H // 2) == d
        r.close()
