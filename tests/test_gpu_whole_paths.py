"""Paths traced whole in one launch against the queue kernels (which run while kernels are timed): the
same images bit for bit and the same ray counts, at chunk sizes around a wave, a block and the sizes
where the choice changes, over chunks of a small pool, several passes and new images.  And traversal
stacks deep enough to spill, against the oracle."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P

pytestmark = pytest.mark.gpu


def _images(scene, W, H, spp, depth, nee, consistent, pool, profile):
    r = P.Renderer(W, H)
    if pool:
        r.set_option(P.OPT_POOL_PATHS, pool)
    r.set_scene(scene)
    r.set_max_depth(depth)
    r.set_nee(nee)
    r.set_option(P.OPT_CONSISTENT_MIS, consistent)
    r.set_option(P.OPT_PROFILE_KERNELS, profile)
    out = []
    for n in (spp, spp + 1, "new", spp):
        if n == "new":
            r.reset()
            continue
        r.render(n)
        out += [r.radiance_sum(), r.radiance(), r.rgba8()]
    st = r.stats()
    out += [np.array(st.bounce_rays), np.array(st.bounce_shadow), st.paths, st.extension_rays, st.shadow_rays]
    assert st.stack_overflows == 0
    r.close()
    return out


@pytest.mark.parametrize("W,H,spp,pool", [(1, 1, 1, 0), (63, 1, 1, 0), (64, 1, 1, 0), (65, 1, 1, 0), (129, 1, 1, 0), (33, 7, 3, 0), (8, 8, 16, 0),
                                          (97, 61, 17, 0), (150, 90, 2, 4096), (1024, 512, 2, 0), (1024, 513, 2, 0)])
@pytest.mark.parametrize("kind", ["cornell", "mesh", "room", "naive"])
def test_whole_paths_equal_the_queues(W, H, spp, pool, kind):
    print(f"case: {kind} {W}x{H}, {spp} spp, pool {pool}", flush=True)
    scene = P.Scene.preset({"mesh": 4, "room": 2}.get(kind, 0), 3, {"mesh": 100000, "room": 100000}.get(kind, 0))
    args = (scene, W, H, spp, {"mesh": 8, "room": 9}.get(kind, 5), kind != "naive", int(kind == "room"), pool)
    for k, (a, b) in enumerate(zip(_images(*args, 0), _images(*args, 1))):
        assert np.array_equal(a, b), k


@pytest.mark.parametrize("lds", [16, 32])
@pytest.mark.parametrize("n", [300, 6000])
def test_spilling_stacks_find_the_closest_hit(n, lds):
    """Long thin triangles through the whole volume: nearly every box holds every ray."""
    print(f"case: {n} long triangles, {lds} stack entries in LDS", flush=True)
    rng = np.random.default_rng(n)
    a = rng.normal(size=(n, 3))
    a /= np.linalg.norm(a, axis=1, keepdims=True)
    side = rng.normal(size=(n, 3)) * 0.02
    off = rng.normal(size=(n, 3)) * 0.3
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
    s.add_triangles(np.concatenate([off - 2 * a, off + 2 * a, off + 2 * a + side], 1), np.full(n, m))
    r = P.Renderer(8, 8)
    r.set_option(P.OPT_TRACE_LDS_STACK, lds)
    r.set_scene(s)
    k = 6000
    org = rng.normal(size=(k, 3)) * 2
    d = off[rng.integers(0, n, k)] - org
    rays = np.concatenate([org, np.zeros((k, 1)), d, np.full((k, 1), 3e38)], 1).astype(np.float32)
    o = O.Scene(s.export(), 8, 8, bvh=True)
    gt, _, _, gp = r.intersect(rays)
    ct, _, _, cp = o.intersect(rays, tri_test=1)
    assert np.array_equal(gp == P.MISS, cp == P.MISS) and (gp != P.MISS).mean() > 0.1
    tie = gp != cp
    assert tie.sum() <= 2 and np.all(np.abs(gt[tie] - ct[tie]) <= 1e-6 * np.abs(ct[tie]))
    shadow = rays.copy()
    shadow[:, 3] = 1e-4
    assert np.array_equal(r.intersect(rays, any_hit=True)[3] == P.MISS, o.intersect(shadow, tri_test=1)[3] == P.MISS)
    assert r.stats().stack_overflows == 0
    r.close()


@pytest.mark.parametrize("W,H", [(128, 128), (128, 129), (256, 128), (257, 128), (256, 256), (362, 362), (512, 257)])
@pytest.mark.parametrize("kind", ["mesh", "room"])
def test_waves_of_few_paths_equal_the_queues(W, H, kind):
    print(f"case: {kind} {W}x{H}", flush=True)
    scene = P.Scene.preset({"mesh": 4, "room": 2}[kind], 3, 100000)
    args = (scene, W, H, 1, 6, True, 0, 0)
    for k, (a, b) in enumerate(zip(_images(*args, 0), _images(*args, 1))):
        assert np.array_equal(a, b), k
