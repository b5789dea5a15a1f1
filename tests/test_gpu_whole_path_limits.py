"""The sizes from which on a pass goes through the queues instead of being traced whole, by the tree's
nodes, its primitives and the estimator: on both sides of each the images and ray counts are the timed
pass's, which always takes the queues.  And whole paths whose waves change columns between their runs."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _soup(n, spheres=False):
    if n == 0:
        return P.Scene.preset(0)   # Cornell box
    rng = np.random.default_rng(n)
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.7, 0.6, 0.5))
    e = s.add_material(P.LAMBERTIAN, (0, 0, 0), (3, 3, 3))
    c = rng.uniform(-2, 2, (n, 3))
    ids = [m if k % 7 else e for k in range(n)]
    if spheres:
        s.add_spheres(c, np.full(n, 0.2), ids)
    else:
        s.add_triangles(np.concatenate([c + 0.6 * rng.normal(size=(n, 3)) for _ in range(3)], 1), ids)
    s.set_camera([0, 0, 6], [0, 0, 0], [0, 1, 0], 0.9)
    return s


def _queues_and_whole(scene, W, H, spp, nee, lds, nodes=(1, 1 << 30)):
    out = []
    for profile in (0, 1):
        r = P.Renderer(W, H)
        r.set_option(P.OPT_TRACE_LDS_STACK, lds)
        r.set_scene(scene)
        r.set_max_depth(4)
        r.set_nee(nee)
        r.set_option(P.OPT_PROFILE_KERNELS, profile)
        r.render(spp)
        st = r.stats()
        out.append([r.radiance_sum(), r.rgba8(), r.path_radiance(W * H * spp), np.array(st.bounce_rays), np.array(st.bounce_shadow)])
        assert nodes[0] <= st.bvh_nodes <= nodes[1] and st.stack_overflows == 0
        r.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    return out[0][0]


@pytest.mark.parametrize("prims,spheres,nee,nodes,limit", [(4, False, 1, (1, 4), 23), (0, False, 1, (1, 4), 23), (40, False, 1, (5, 16), 21),
                                                           (300, False, 1, (17, 1000), 21), (300, False, 0, (17, 1000), 20.585), (300, True, 1, (17, 1000), 20)])
@pytest.mark.parametrize("above", [0, 1])
@pytest.mark.parametrize("lds", [16, 32])
def test_both_sides_of_a_limit(prims, spheres, nee, nodes, limit, above, lds):
    W = 1 << int(limit + 1) // 2
    H = round(2 ** limit) // W + above
    print(f"case: {prims} {'spheres' if spheres else 'triangles'}, nee {nee}, {W}x{H}, {lds} stack rows", flush=True)
    image = _queues_and_whole(_soup(prims, spheres), W, H, 1, nee, lds, nodes)
    assert prims == 4 or image.any()   # (the one light of the four faces away)


@pytest.mark.parametrize("W,H,spp", [(1024, 512, 8), (512, 1024, 3), (700, 1500, 1), (333, 777, 5), (1024, 512, 2), (768, 512, 1), (2048, 64, 5)])
@pytest.mark.parametrize("prims", [0, 300])
@pytest.mark.parametrize("lds", [16, 32])
def test_waves_that_change_columns_trace_every_path(W, H, spp, prims, lds):
    print(f"case: {prims} triangles, {W}x{H}x{spp}, {lds} stack rows", flush=True)
    assert _queues_and_whole(_soup(prims), W, H, spp, 1, lds).any()
