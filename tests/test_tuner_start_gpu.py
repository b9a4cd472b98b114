"""The tuner's search starts from the configuration an untuned tracer runs with, so that tuning never
replaces it by a slower one, and what it finds for passes that overlap leaves a pass alone as it was.
The bounds are wide for timings: run-to-run differences are a few percent, a search from the
library's base configuration is off by 40% (its start) and 13% (a pass alone)."""
import statistics
import time

import numpy as np
import pytest

import exposure_render as er
from exposure_render import scenes

pytestmark = pytest.mark.gpu


def _scene(w, h):
    sc = scenes.config_ct(scale=0.5, bilateral=False)
    sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = w, h
    return sc


def _overlapped(r):
    return min(r.render_passes(16).total_ms / 16 for _ in range(8))


def _alone(r):
    """a pass alone, ms: the best of five medians, so that a busy host does not count"""
    medians = []
    for _ in range(5):
        times = []
        for _ in range(20):
            a = time.perf_counter()
            r.render_estimate()
            times.append(time.perf_counter() - a)
        medians.append(statistics.median(times))
    return min(medians) * 1e3


@pytest.mark.parametrize("film", [(360, 340), (640, 480)])
def test_tuning_starts_from_what_runs(fresh, film):
    sc = _scene(*film)
    r = er.Renderer(sc, seed=4)
    _overlapped(r)
    untuned, alone = _overlapped(r), _alone(r)
    t = r.autotune(passes=16, force=True)
    tuned, after = _overlapped(r), _alone(r)
    print(f"[tune] {film} a pass {untuned:.3f} ms untuned, {tuned:.3f} tuned, alone {alone:.3f}, {after:.3f} {t}", flush=True)
    assert t["default_ms_per_pass"] <= 1.2 * untuned
    assert tuned <= 1.1 * untuned
    assert after <= 1.08 * alone
    r.rebind()
    r.seed(6)
    r.render_passes(2)
    f = er.Renderer(sc, seed=6)
    f.render_passes(2)
    assert np.array_equal(r.frame(), f.frame())
    r.close()
    f.close()


def test_batch_tuning_starts_from_what_runs(fresh):
    """Jobs of different bricks (one is clipped) start the search with their own. What it finds holds
    for the jobs' later passes, bricks included, so nothing is asked of passes outside a batch."""
    scs = [_scene(256, 256), _scene(200, 180)]
    scs[1].add_clip(scenes.clipping_box((0.3, 0.0, 0.0), (0.4, 1.1, 1.1)))
    rs = [er.Renderer(sc, seed=4) for sc in scs]
    untuned = min(er.render_batch(rs, [8, 8]).total_ms / 8 for _ in range(8))
    t = er.autotune_batch(rs, rounds=8)
    print(f"[tune] batch round {untuned:.3f} ms untuned {t}", flush=True)
    assert t["default_ms_per_pass"] <= 1.2 * untuned
    assert t["ms_per_pass"] <= t["default_ms_per_pass"] and t["brick"] in (2, 4, 8, 16, 32)
    for r, sc in zip(rs, scs):
        r.rebind()
        r.seed(6)
    er.render_batch(rs, [2, 2])
    for r, sc in zip(rs, scs):
        f = er.Renderer(sc, seed=6)
        f.render_passes(2)
        assert np.array_equal(r.frame(), f.frame())
        f.close()
        r.close()


def test_a_given_configuration_holds_for_every_pass(fresh):
    """er_set_tune is taken as given; a later search is free to move on from it."""
    r = er.Renderer(_scene(256, 256), seed=4)
    base = dict(r.get_tune())
    r.render_passes(2)
    assert r.get_tune() == base and (base["brick"], base["blocks_per_cu"], base["heavy_tiles"]) == (8, 7, 0)
    r.set_tune(8, 8, 5, 2, 0, 4, 16, 4)
    r.render_estimate()
    t = r.get_tune()
    assert (t["blocks_per_cu"], t["shadow_waves_per_cu"], t["rays_per_wave"], t["shadow_rays_per_wave"]) == (5, 2, 4, 16)
    s = r.autotune(passes=2, force=True)
    assert s["ms_per_pass"] <= s["default_ms_per_pass"]
    t = r.get_tune()
    assert all(t[k] == s[k] for k in ("brick", "tile_w", "blocks_per_cu", "shadow_waves_per_cu", "heavy_tiles", "rays_per_wave"))
    r.close()
