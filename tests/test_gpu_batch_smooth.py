"""Scenes with per-vertex normals among the renders of a batch: the images are those of the same renders on
their own, whatever the other renders' scenes have, with the scenes' emitters smooth or flat."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _scene(k, kind):
    rng = np.random.default_rng(k)
    s = P.Scene()
    ids = [s.add_material(P.LAMBERTIAN, (0.6, 0.5, 0.4)), s.add_material(P.LAMBERTIAN, (0.4, 0.4, 0.4), emit=(3, 2, 1))]
    n = 61 + 40 * k
    c = rng.normal(size=(n, 3))
    tri = np.concatenate([c + 0.5 * rng.normal(size=(n, 3)) for _ in range(3)], 1)
    normals = None
    if kind != "flat":
        normals = rng.normal(size=(n, 9))
        if kind == "mixed":   # every other triangle's normals are the flat one
            a, b, d = (tri[::2, 3 * j:3 * j + 3] for j in range(3))
            normals[::2] = np.tile(np.cross(b - a, d - a), 3)
    s.add_triangles(tri, np.where(np.arange(n) % 9 == 0, ids[1], ids[0]), normals=normals)
    s.set_environment(rng.uniform(0.1, 2, (8, 16, 4)).astype(np.float32))
    s.set_camera([0, 0.2, 4], [0, 0, 0], [0, 1, 0], 0.9)
    return s


@pytest.mark.parametrize("kinds", [("smooth",), ("flat", "smooth"), ("smooth", "smooth", "smooth"), ("flat", "flat", "mixed", "smooth", "flat", "mixed")])
@pytest.mark.parametrize("W,H,spp", [(33, 21, 3), (160, 120, 4)])
def test_batch_of_scenes_with_vertex_normals(kinds, W, H, spp):
    print(f"case: {kinds}, {W}x{H}, {spp} spp", flush=True)
    b = P.Batch()
    want = []
    for k, kind in enumerate(kinds):
        s = _scene(k, kind)
        b.add(s, W, H, spp, 4)
        r = P.Renderer(W, H)
        r.set_scene(s)
        r.set_max_depth(4)
        r.render(spp)
        want.append(r.radiance())
        r.close()
    for _ in range(3):
        b.run()
        for k in range(len(kinds)):
            assert np.array_equal(b.radiance(k), want[k]), k
    b.close()
