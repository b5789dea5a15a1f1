"""The sizes from which on a pass goes through the queues instead of being traced whole, by the tree's
nodes: on both sides of each the images and ray counts are the timed pass's, which always takes the queues."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _soup(n):
    if n == 0:
        return P.Scene.preset(0)   # Cornell box
    rng = np.random.default_rng(n)
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.7, 0.6, 0.5))
    e = s.add_material(P.LAMBERTIAN, (0, 0, 0), (3, 3, 3))
    c = rng.uniform(-2, 2, (n, 3))
    s.add_triangles(np.concatenate([c + 0.6 * rng.normal(size=(n, 3)) for _ in range(3)], 1), [m if k % 7 else e for k in range(n)])
    s.set_camera([0, 0, 6], [0, 0, 0], [0, 1, 0], 0.9)
    return s


@pytest.mark.parametrize("prims,nodes,limit", [(4, (1, 4), 22), (0, (1, 4), 22), (40, (5, 16), 21), (300, (17, 1000), 20)])
@pytest.mark.parametrize("above", [0, 1])
@pytest.mark.parametrize("lds", [16, 32])
def test_both_sides_of_a_limit(prims, nodes, limit, above, lds):
    W, H = 1 << (limit + 1) // 2, (1 << limit // 2) + above
    print(f"case: {prims} triangles, {W}x{H}, {lds} stack rows", flush=True)
    scene = _soup(prims)
    out = []
    for profile in (0, 1):
        r = P.Renderer(W, H)
        r.set_option(P.OPT_TRACE_LDS_STACK, lds)
        r.set_scene(scene)
        r.set_max_depth(4)
        r.set_option(P.OPT_PROFILE_KERNELS, profile)
        r.render(1)
        st = r.stats()
        out.append([r.radiance_sum(), r.rgba8(), np.array(st.bounce_rays), np.array(st.bounce_shadow)])
        assert nodes[0] <= st.bvh_nodes <= nodes[1] and st.stack_overflows == 0
        r.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert prims == 4 or out[0][0].any()   # (the one light of the four faces away)
