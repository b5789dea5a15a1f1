"""Picks and the normals view at window sizes around the view's 8 x 8 pixel tiles, against the oracle's
intersections of the pixel-centre rays."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P

pytestmark = pytest.mark.gpu


def _scene():
    s = P.Scene.preset(4, seed=2, param=5000)
    s.add_spheres([[0.9, 0.6, 1.0], [-1.2, -0.4, 0.8]], [0.3, 0.25], [0, 1])
    # off the mesh's plane of symmetry, whose rays run along shared edges
    s.set_camera([0.117, 0.293, 3.2], [0.031, -0.012, 0.0], [0.0, 1.0, 0.0], 0.7)
    return s


def _centre_rays(cam, W, H):
    """camera.cu:24-27: pixel-centre rays of a camera looking from its origin to its target."""
    o, t, up = (np.asarray(cam[k], np.float64) for k in ("origin", "target", "up"))
    z = (o - t) / np.linalg.norm(o - t)
    x = np.cross(up / np.linalg.norm(up), z)
    x /= np.linalg.norm(x)
    y = np.cross(z, x)
    top = np.tan(cam["vfov"] / 2)
    c, r = np.meshgrid((np.arange(W) + 0.5) / W, (np.arange(H) + 0.5) / H)
    d = (2 * c - 1)[..., None] * (top * W / H) * x + (2 * r - 1)[..., None] * top * y - z
    d /= np.linalg.norm(d, axis=-1, keepdims=True)
    n = W * H
    return np.concatenate([np.tile(o, (n, 1)), np.zeros((n, 1)), d.reshape(n, 3), np.full((n, 1), 3e38)], 1).astype(np.float32)


@pytest.mark.parametrize("lds", [16, 32])
@pytest.mark.parametrize("W,H", [(1, 1), (7, 9), (8, 8), (9, 7), (65, 33), (160, 100)])
def test_normals_and_picks_match_the_oracle(W, H, lds):
    print(f"case: {W}x{H}, {lds} stack entries in LDS", flush=True)
    s = _scene()
    a = s.export()
    r = P.Renderer(W, H)
    r.set_option(P.OPT_TRACE_LDS_STACK, lds)
    r.set_scene(s)
    rays = _centre_rays(a["camera"], W, H)
    t, _, _, prim = O.Scene(a, W, H, bvh=True).intersect(rays, tri_test=1)
    nt = len(a["tri_pos"])
    v = a["tri_pos"].reshape(nt, 3, 3).astype(np.float64)
    tri = np.clip(prim, 0, nt - 1)
    n = np.cross(v[tri, 1] - v[tri, 0], v[tri, 2] - v[tri, 0])
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    mat = a["tri_mat"][tri].copy()
    for k, (sph, m) in enumerate(zip(a["sph"], a["sph_mat"])):
        of = prim == ~k
        n[of] = (rays[of, :3] + rays[of, 4:7] * t[of, None] - sph[:3]) / sph[3]
        mat[of] = m
    miss = prim == P.MISS
    want = np.where(miss[:, None], 0.0, (n + 1) / 2)
    r.set_type(P.RENDERER_NORMALS)
    # a last-bit difference between the two sets of rays may move a ray across an edge: the rest agree
    for passes in (1, 2):
        r.render(1)
        got = r.radiance().reshape(-1, 3)
        assert (np.abs(got - want).max(1) < 1e-4).mean() >= 1 - max(2, 0.002 * W * H) / (W * H)
        sums = r.radiance_sum().reshape(-1, 3)
        assert np.array_equal((sums / passes).astype(np.float32), got)
    r.set_option(P.OPT_TRACE_STATS, 1)
    r.reset()
    r.reset_stats()
    r.render(1)
    assert np.array_equal(r.radiance().reshape(-1, 3), got) and r.stats().trace_rays[0] == W * H
    rng = np.random.default_rng(1)
    wrong = 0
    for p in rng.integers(0, W * H, 24):
        m, hit = r.hit_test(int(p % W), int(p // W))
        wrong += (hit, m) != ((False, -1) if miss[p] else (True, int(mat[p])))
    assert wrong <= 1
    assert r.hit_test(W, 0) == (-1, False) and r.hit_test(-1, 0) == (-1, False)
    r.close()
