"""A tracer keeps its opacity table, occupancy bits, majorants and the volume's gradient maximum
from bind to bind and rebuilds them when what they were built from changes. Each change below is
made to a tracer that has rendered, and the next passes must be those of a tracer bound fresh with
the changed scene, bit for bit - and again after the change is undone."""
import ctypes as C

import numpy as np
import pytest

import exposure_render as er
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _scene():
    sc = scenes.config_ct(scale=0.2, bilateral=True)
    sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = 90, 70
    sc.add_clip(scenes.clipping_box((0.3, 0.0, 0.0), (0.4, 1.1, 1.1)))
    return sc


def _passes(r):
    r.seed(11)
    r.render_passes(2)
    return r.frame(), r.get_seeds(), r.get_estimate()


def _bind(r, kind):
    fn = {"tracer": r.lib.er_bind_tracer, "volume": r.lib.er_bind_volume, "clip": r.lib.er_bind_clipping_object}[kind]
    d = {"tracer": r.tracer, "volume": r.volume, "clip": r.clips[0]}[kind]
    if kind == "tracer":
        d.no_iterations = 0
    assert fn(C.byref(d), 1) == capi.ER_OK


def _opacity(d):
    d.opacity.init()
    d.opacity.add(0.0, 0.0).add(500.0, 0.0).add(900.0, 0.3).add(4095.0, 0.2)


def _set(**kw):
    def change(d):
        for k, v in kw.items():
            setattr(d.settings, k, v)
    return change


def _camera(d):
    d.camera.pos[0], d.camera.pos[2] = -1.4, 1.3


def _spacing(d):
    d.spacing[1] = 1.7


def _clip(d):
    d.shape.inv_tm[0][3] = 0.25
    d.shape.tm[0][3] = -0.25


CHANGES = {
    "camera": ("tracer", _camera), "opacity": ("tracer", _opacity), "density": ("tracer", _set(density_scale=30.0)),
    "compat": ("tracer", _set(estimator=capi.ESTIMATOR_COMPAT)), "woodcock": ("tracer", _set(sampler=capi.SAMPLER_WOODCOCK)),
    "phase": ("tracer", _set(shading_type=capi.SHADING_PHASE_ONLY)),
    "filter": ("tracer", _set(bilateral_radius=5, bilateral_sigma_range=9.0)),
    "spacing": ("volume", _spacing), "clip": ("clip", _clip), "voxels": ("volume", None),
}


@pytest.mark.parametrize("change", sorted(CHANGES))
def test_a_changed_bind_renders_as_a_fresh_one(fresh, change):
    kind, edit = CHANGES[change]
    print(f"[rebind] {change}", flush=True)
    sc = _scene()
    other = np.ascontiguousarray(sc.voxels[::-1, :, ::-1] // 2)
    fresh_sc = _scene()
    if change == "voxels":
        fresh_sc.voxels[:] = other
    else:
        edit({"tracer": fresh_sc.tracer, "volume": fresh_sc.volume, "clip": fresh_sc.clips[0]}[kind])
    f = er.Renderer(fresh_sc)
    want = _passes(f)
    f.close()

    r = er.Renderer(sc)
    base = _passes(r)
    d = {"tracer": r.tracer, "volume": r.volume, "clip": r.clips[0]}[kind]
    before = type(d).from_buffer_copy(d)
    before.id = d.id
    if change == "voxels":           # new contents at the same address
        kept = sc.voxels.copy()
        sc.voxels[:] = other
        d.voxels_dirty = 1
    else:
        edit(d)
    _bind(r, kind)
    r.rebind()
    got = _passes(r)
    C.memmove(C.byref(d), C.byref(before), C.sizeof(d))
    if change == "voxels":
        sc.voxels[:] = kept
        d.voxels_dirty = 1
    _bind(r, kind)
    r.rebind()
    again = _passes(r)
    r.close()
    for x, y in ((got, want), (again, base)):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[2], y[2])
        assert np.array_equal(x[1][0], y[1][0]) and np.array_equal(x[1][1], y[1][1])
    assert not np.array_equal(base[2], want[2])


def test_node_table_on_and_off(fresh):
    sc = scenes.config_adjoint(scale=0.25)
    r = er.Renderer(sc)
    base = _passes(r)
    images = []
    for seed in (1, 2, 1):
        r.set_tf_lut(scenes.random_tf_lut(seed), sc.tf_range)
        images.append(_passes(r)[0])
    assert np.array_equal(images[0], images[2]) and not np.array_equal(images[0], images[1])
    r.set_tf_lut(None, 0.0)
    assert np.array_equal(_passes(r)[0], base[0])
    r.close()


def test_adjoint_workspace_follows_the_film(fresh):
    """er_adjoint_lut keeps its buffers with the tracer: repeated calls, and calls after the film
    grew and shrank, give the gradient of a fresh tracer (sums of float atomics: to rounding)."""
    sc = scenes.config_adjoint(scale=0.25)
    lut = scenes.initial_tf_lut()
    rng = np.random.default_rng(3)

    def gradient(r, w, h):
        s1, s2 = er.seeds_for(w, h, 5)
        return r.adjoint_lut(s1, s2, 3, g[(w, h)])
    sizes = [(64, 48), (130, 70), (20, 31), (64, 48)]
    g = {s: rng.normal(size=(s[1], s[0], 3)).astype(np.float32) for s in sizes}
    want = {}
    for w, h in set(sizes):
        sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = w, h
        f = er.Renderer(sc)
        f.set_tf_lut(lut, sc.tf_range)
        want[(w, h)] = gradient(f, w, h)
        f.close()
    r = er.Renderer(sc)
    r.set_tf_lut(lut, sc.tf_range)
    for w, h in sizes:
        r.tracer.camera.film_size[0], r.tracer.camera.film_size[1] = w, h
        r.rebind()
        r.W, r.H = w, h
        for _ in range(2):
            got = gradient(r, w, h)
            assert np.abs(got - want[(w, h)]).max() <= 2e-5 * np.abs(want[(w, h)]).max()
    r.close()


def _nothing(v):
    v.resolution[0], v.resolution[2] = 4 * v.resolution[0], 3 * v.resolution[2]
    v.voxels = None


def _empty(v):
    v.resolution[1] = 0


def _too_large(v):
    v.resolution[0] = v.resolution[1] = 1 << 13
    v.resolution[2] = 1


@pytest.mark.parametrize("edit", [_nothing, _empty, _too_large])
def test_a_refused_volume_leaves_the_bound_one(fresh, edit):
    """A rebind that is refused changes nothing: the next binds and passes see the volume as it was,
    its size with its buffers, and a later good rebind takes its place."""
    print(f"[rebind] refused: {edit.__name__}", flush=True)
    sc = _scene()
    r = er.Renderer(sc)
    base = _passes(r)
    v = r.volume
    kept = [v.resolution[i] for i in range(3)]
    v.spacing[0] = 3.0
    edit(v)
    v.voxels_dirty = 1
    assert r.lib.er_bind_volume(C.byref(v), 1) == capi.ER_ERROR
    r.rebind()
    again = _passes(r)
    for i in range(3):
        v.resolution[i] = kept[i]
    v.spacing[0] = 1.0
    other = np.ascontiguousarray(sc.voxels[::-1, :, ::-1] // 2)
    v.voxels = other.ctypes.data_as(C.POINTER(C.c_uint16))
    _bind(r, "volume")
    r.rebind()
    got = _passes(r)
    r.close()
    sc.voxels[:] = other
    f = er.Renderer(sc)
    want = _passes(f)
    f.close()
    for x, y in ((again, base), (got, want)):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[2], y[2])
        assert np.array_equal(x[1][0], y[1][0]) and np.array_equal(x[1][1], y[1][1])
    assert not np.array_equal(base[2], want[2])


def test_display_filter_follows_each_bind(fresh):
    """The filter's tables are rebuilt by the bind that changes them and read by the pass that
    follows at once, on the tracer's streams."""
    sc = _scene()
    r = er.Renderer(sc)
    for radius, spatial, rng in [(2, 1.5, 20.0), (7, 4.0, 60.0), (0, 1.0, 1.0), (32, 9.0, 30.0), (2, 1.5, 20.0)]:
        print(f"[rebind] filter {radius} {spatial} {rng}", flush=True)
        images = []
        for d in (r.tracer, sc.tracer):
            d.settings.bilateral_radius, d.settings.bilateral_sigma_spatial, d.settings.bilateral_sigma_range = radius, spatial, rng
        r.rebind()
        f = er.Renderer(sc)
        for x in (r, f):
            images.append(_passes(x)[2])
        f.close()
        assert np.array_equal(*images)
    r.close()


@pytest.mark.parametrize("tuned", [False, True])
def test_clipping_object_comes_and_goes(fresh, tuned):
    """A kept tracer changes march form, and untuned its bricks, when its clipping object is added
    to it, taken from it or unbound; each time it renders as a tracer bound fresh."""
    def scene(clip):
        sc = scenes.config_ct(scale=0.2, bilateral=True)
        sc.tracer.camera.film_size[0], sc.tracer.camera.film_size[1] = 90, 70
        if clip:
            sc.add_clip(scenes.clipping_box((0.3, 0.0, 0.0), (0.4, 1.1, 1.1)))
        return sc

    def passes(r):
        if tuned:
            r.set_tune(4, 8, 4, 4, 64, 64, 64, 16)
        out = _passes(r)
        r.seed(7)
        r.render_estimate()
        return out + (r.frame(),)
    want = {}
    for clip in (False, True):
        f = er.Renderer(scene(clip))
        want[clip] = passes(f)
        f.close()
    assert not np.array_equal(want[False][2], want[True][2])
    r = er.Renderer(scene(True))
    ident = r.tracer.clipping_ids[0]
    for clip, count, bound in [(True, 1, True), (False, 0, True), (True, 1, True), (False, 1, False)]:
        print(f"[rebind] clipping object: listed {count} bound {bound} tuned {tuned}", flush=True)
        r.tracer.clipping_count, r.tracer.clipping_ids[0] = count, ident
        if not bound:
            assert r.lib.er_bind_clipping_object(C.byref(r.clips[0]), 0) == capi.ER_OK
        r.rebind()
        got = passes(r)
        assert all(np.array_equal(a, b) for a, b in zip((got[0], got[2], got[3]), (want[clip][0], want[clip][2], want[clip][3])))
        assert all(np.array_equal(a, b) for a, b in zip(got[1], want[clip][1]))
    r.close()


@pytest.mark.parametrize("film", [(-3, 70), (90, -1)])
def test_a_refused_film_leaves_the_bound_tracer(fresh, film):
    """A rebind whose film is refused changes nothing, its other settings included."""
    print(f"[rebind] refused film {film}", flush=True)
    r = er.Renderer(_scene())
    base = _passes(r)
    t = r.tracer
    kept = type(t).from_buffer_copy(t)
    t.camera.film_size[0], t.camera.film_size[1] = film
    t.settings.density_scale = 1.0
    assert r.lib.er_bind_tracer(C.byref(t), 1) == capi.ER_ERROR
    _bind(r, "clip")                 # a bind of something else: parameters are built again
    r.seed(11)
    r.render_passes(2)               # passes 3 and 4 of the tracer as it was
    got = r.frame(), r.get_seeds()
    assert r.no_iterations() == 4
    assert np.array_equal(got[0], base[0])
    assert np.array_equal(got[1][0], base[1][0]) and np.array_equal(got[1][1], base[1][1])
    C.memmove(C.byref(t), C.byref(kept), C.sizeof(t))
    r.rebind()
    again = _passes(r)
    r.close()
    assert np.array_equal(again[0], base[0])
