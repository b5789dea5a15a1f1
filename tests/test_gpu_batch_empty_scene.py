"""Renders of an environment alone, without primitives, among the renders of a batch: the images are those
of the same renders on their own, in first, middle and last place, with one launch and with two per bounce."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _scene(k, empty):
    rng = np.random.default_rng(k)
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.6, 0.5, 0.4))
    if not empty:
        c = rng.normal(size=(300, 3))
        s.add_triangles(np.concatenate([c + 0.4 * rng.normal(size=(300, 3)) for _ in range(3)], 1), np.full(300, m))
    s.set_environment(rng.uniform(0.1, 2, (8, 16, 4)).astype(np.float32))
    s.set_camera([0, 0.2, 4], [0, 0, 0], [0, 1, 0], 0.9)
    return s


@pytest.mark.parametrize("empty", [(0,), (1,), (2,), (0, 2), (0, 1, 2)])
@pytest.mark.parametrize("W,H,spp", [(33, 21, 3), (160, 120, 4)])
def test_batch_with_scenes_without_primitives(empty, W, H, spp):
    print(f"case: renders {empty} of 3 without primitives, {W}x{H}, {spp} spp", flush=True)
    b = P.Batch()
    want = []
    for k in range(3):
        s = _scene(k, k in empty)
        b.add(s, W, H, spp, 4)
        r = P.Renderer(W, H)
        r.set_scene(s)
        r.set_max_depth(4)
        r.render(spp)
        want.append(r.radiance())
        r.close()
    for _ in range(3):
        b.run()
        for k in range(3):
            assert np.array_equal(b.radiance(k), want[k]), k
    assert b.stats()["stack_overflows"] == 0
    b.close()
