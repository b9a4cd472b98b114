"""er_adjoint_lut over its pass pipeline and its marches' forms.

Passes go round a few buffer sets, each with a gradient sum and a stream of its own: from one pass
(sets left unused) to several rounds, on films from one pixel to ragged ones, the gradient must be
er_adjoint_lut_noalloc's, which runs the same kernels one pass after the other. Scenes with
clipping objects take the marches' general form and others the plain one: an object that clips
nothing must not change the gradient. Both sides add the same FP32 terms in another order: 1e-4
relative per entry, plus 1e-5 of the largest entry for entries whose terms cancel."""
import numpy as np
import pytest

import exposure_render as er
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _lut(kind):
    lut = scenes.initial_tf_lut().copy()
    if kind == "positive":      # no empty cells: every sample counts
        lut[:, 0] = np.linspace(0.02, 0.6, lut.shape[0])
    elif kind == "sparse":      # most cells empty
        lut[:, 0] = np.maximum(0.0, np.linspace(-2.0, 0.8, lut.shape[0]))
    return lut


def _renderer(w, h, kind, clip=False):
    sc = scenes.config_adjoint(scale=0.25)
    sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = w, h
    if clip:
        tm, inv = scenes.translate((9.0, 0.0, 0.0))
        sc.add_clip(scenes.clipping_shape(capi.SHAPE_BOX, tm, inv, size=(0.1, 0.1, 0.1)))
    r = er.Renderer(sc)
    r.set_tf_lut(_lut(kind), sc.tf_range)
    return r


def _close(got, want):
    scale = np.abs(want).max()
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - want) <= 1e-4 * np.abs(want) + 1e-5 * scale)


@pytest.mark.parametrize("w,h,passes,kind", [
    (1, 1, 2, "positive"), (65, 3, 1, "positive"), (7, 41, 3, "sparse"), (64, 64, 4, "initial"),
    (129, 67, 7, "positive"), (130, 65, 6, "sparse"), (256, 100, 5, "initial")])
def test_passes_and_forms(w, h, passes, kind, fresh):
    s1, s2 = er.seeds_for(w, h, 17)
    A = np.random.default_rng(w + h).standard_normal((h, w, 3)).astype(np.float32)
    r = _renderer(w, h, kind)
    got = [r.adjoint_lut(s1, s2, passes, A) for _ in range(2)]   # (also uploads the device's tables)
    want = r.adjoint_lut_noalloc(s1, s2, passes, A)
    print(f"[adjoint-passes] {w}x{h} passes {passes} {kind}: max |g| {np.abs(want).max():.3e}", flush=True)
    _close(got[0], want)
    _close(got[1], want)
    clipped = _renderer(w, h, kind, clip=True)
    _close(clipped.adjoint_lut(s1, s2, passes, A), want)
