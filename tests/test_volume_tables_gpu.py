"""The tables the device derives from a volume - cell records and largest voxel, macrocell ranges,
occupancy bits, group radii, gradient-magnitude maximum - at sizes that leave remainders of the
bricks (2 to 32 cells), of the groups of 4 bricks and of a cell column's run: a macrocell wrongly
taken for empty, a radius too large or a wrong record changes the image, which the oracle renders
without any of them."""
import numpy as np
import pytest

import exposure_render as er
import oracle as O
from exposure_render import capi, scenes

pytestmark = pytest.mark.gpu


def _scene(shape, peak, spacing):
    """Isolated voxels and one plateau in an otherwise empty volume, so that most bricks are
    empty and the occupied ones lie anywhere, the faces included."""
    rz, ry, rx = shape
    rng = np.random.default_rng(rz * 10007 + ry * 101 + rx)
    vox = np.zeros(shape, dtype=np.uint16)
    n = max(2, vox.size // 400)
    vox.reshape(-1)[rng.integers(0, vox.size, n)] = rng.integers(peak // 4, peak + 1, n)
    vox[rz // 2:rz // 2 + 2, ry // 2:ry // 2 + 2, :max(1, rx // 3)] = peak
    vox[-1, -1, -1] = peak
    sc = scenes.config_ct(scale=0.1, bilateral=False)
    base = scenes.Scene(vox, spacing)
    sc.voxels, sc.volume = base.voxels, base.volume
    t = sc.tracer
    t.opacity.init()
    t.opacity.add(0.0, 0.0).add(peak / 5.0, 0.0).add(peak / 2.0, 0.2).add(float(peak), 1.0)
    t.camera.film_size[0], t.camera.film_size[1] = 61, 47
    return sc


@pytest.mark.parametrize("shape,peak,spacing,bricks", [
    ((1, 1, 1), 4000, (1.0, 1.0, 1.0), (2, 8)),
    ((2, 3, 5), 4095, (1.0, 1.0, 1.0), (2, 4, 8)),
    ((8, 8, 8), 4095, (1.0, 1.0, 1.0), (2, 8)),
    ((9, 31, 17), 4095, (1.0, 0.7, 1.3), (2, 4, 16)),
    ((33, 16, 67), 65535, (1.0, 1.0, 1.0), (4, 8, 32)),
    ((70, 5, 129), 300, (0.5, 1.0, 1.0), (2, 8, 32)),
])
def test_odd_volumes_render_as_without_tables(fresh, shape, peak, spacing, bricks):
    sc = _scene(shape, peak, spacing)
    orc = O.Oracle(sc)
    gm_ref = orc.compute_gm_max()
    seeds = O.seeds_for(61, 47, 3)
    s1, s2 = seeds[0].copy(), seeds[1].copy()
    frames = [orc.trace(s1, s2)[0] for _ in range(2)]
    for brick in bricks:
        print(f"[tables] shape={shape} brick={brick}", flush=True)
        r = er.Renderer(sc)
        r.set_tune(brick, 8, 7)
        r.set_seeds(*seeds)
        assert r.gm_max() == gm_ref
        for f_ref in frames:
            r.render_estimate()
            f = r.frame()
            assert np.array_equal(f[..., 3], f_ref[..., 3])
            np.testing.assert_allclose(f, f_ref, rtol=1e-4, atol=1e-6)
        g1, g2 = r.get_seeds()
        assert np.array_equal(g1, s1) and np.array_equal(g2, s2)
        r.close()
