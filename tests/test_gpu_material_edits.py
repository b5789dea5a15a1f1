"""Material edits on scenes on both sides of the one-block emitter list: the image after an edit is that of
a scene loaded with the edited materials, bit for bit, for edits that add, change and remove emission, change
the type, and leave a colour as it was."""
import ctypes as C

import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _scene(n, mats):
    rng = np.random.default_rng(n)
    s = P.Scene()
    ids = [s.add_material(*m) for m in mats]
    if n:
        c = rng.uniform(-2, 2, (n, 1, 3))
        s.add_triangles((c + rng.normal(size=(n, 3, 3)) * max(0.05, 1.5 / n ** 0.5)).reshape(n, 9), [ids[k] for k in rng.integers(0, len(ids), n)])
    s.add_spheres(rng.uniform(-2, 2, (4, 3)), np.full(4, 0.3), [ids[k % len(ids)] for k in range(4)])
    s.set_environment(np.full((2, 4, 4), 0.2, np.float32))
    s.set_camera([0, 0.1, 7], [0, 0, 0], [0, 1, 0], 0.8)
    return s


def _image(r):
    r.render(3)
    return r.radiance_sum()


@pytest.mark.parametrize("n", [0, 1, 1019, 1020, 1021, 2043, 2044, 2045, 5000])
def test_edits_equal_a_load(n):
    print(f"case: {n} triangles and 4 spheres", flush=True)
    L = P.LAMBERTIAN
    mats = [(L, (0.6, 0.5, 0.4), (0, 0, 0)), (L, (0, 0, 0), (3, 2, 1)), (L, (0.3, 0.6, 0.5), (0, 0, 0)), (P.GLASS, (0, 0, 0), (0, 0, 0), 1.5)]
    r = P.Renderer(48, 40)
    r.set_scene(_scene(n, mats))
    r.set_max_depth(5)
    for k, to in ((0, (L, (0.6, 0.5, 0.4), (1, 2, 3))), (1, (L, (0, 0, 0), (0.5, 2, 1))), (2, (L, (0.2, 0.7, 0.1), (0, 0, 0))),
                  (3, (L, (0.5, 0.5, 0.5), (2, 2, 2))), (1, (P.MIRROR, (1, 1, 1), (0.5, 2, 1))), (3, (P.MICROFACET, (1, 1, 1), (0, 0, 0), 1.3, 0.2)),
                  (0, (L, (0.6, 0.5, 0.4), (0, 0, 0)))):
        mats[k] = to
        r.set_material(k, *to)
        w = P.Renderer(48, 40)
        w.set_scene(_scene(n, mats))
        w.set_max_depth(5)
        assert np.array_equal(_image(r), _image(w)), (k, to)
        w.close()
    # null colours stay
    e = np.array([4, 1, 1], np.float32)
    P.check(P.lib().pt_renderer_set_material(r.h, 2, L, None, e.ctypes.data_as(C.c_void_p), 1.5, 0.1))
    mats[2] = (L, (0.2, 0.7, 0.1), (4, 1, 1), 1.5, 0.1)
    w = P.Renderer(48, 40)
    w.set_scene(_scene(n, mats))
    w.set_max_depth(5)
    assert np.array_equal(_image(r), _image(w))
    P.check(P.lib().pt_renderer_set_material(r.h, 2, L, None, None, 1.5, 0.1))
    r.reset()
    w.reset()
    assert np.array_equal(_image(r), _image(w))
    r.close()
    w.close()
