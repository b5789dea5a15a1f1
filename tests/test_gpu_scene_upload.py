"""Scene uploads at the sizes where the build on the device changes shape: one primitive, the leaf
size, the tile of leaves a workgroup climbs, the largest one-block sort and one past each, a tree of
two climbs, and trees without any extent; then the emitter list and the kept per-vertex normals, made
on the device in input order."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P
from helpers import path_agreement

pytestmark = pytest.mark.gpu


def _scene(n, rng, same=False):
    c = np.zeros((n, 3)) if same else rng.uniform(-2, 2, (n, 3))
    e = rng.normal(size=(1 if same else n, 3, 3)) * (0.5 if same else max(0.02, 2.0 / n ** (1 / 2)))
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
    s.add_triangles((c[:, None, :] + e).reshape(n, 9), np.full(n, m))
    return s


@pytest.mark.parametrize("builder", [P.BVH_LBVH, P.BVH_PLOC])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 1023, 1024, 1025, 2047, 2048, 2049, 65536, 65537])
def test_closest_hits_at_build_edges(n, builder):
    print(f"case: {n} triangles, builder {builder}", flush=True)
    rng = np.random.default_rng(n)
    s = _scene(n, rng)
    r = P.Renderer(8, 8)
    r.set_option(P.OPT_BVH_BUILDER, builder)
    r.set_scene(s)
    o = O.Scene(s.export(), 8, 8, bvh=True)
    org = rng.uniform(-4, 4, (4000, 3))
    at = s.export()["tri_pos"].reshape(n, 3, 3).mean(1)[rng.integers(0, n, 4000)]
    rays = np.concatenate([org, np.zeros((4000, 1)), at - org, np.full((4000, 1), 3e38)], 1).astype(np.float32)
    gt, _, _, gp = r.intersect(rays)
    ct, _, _, cp = o.intersect(rays, tri_test=1)
    # every ray aims at a triangle's centre; where two triangles tie, the distances are the same
    assert np.array_equal(gp == P.MISS, cp == P.MISS) and (gp != P.MISS).mean() > 0.99
    tie = gp != cp
    assert tie.sum() <= 2 and np.all(np.abs(gt[tie] - ct[tie]) <= 1e-6 * np.abs(ct[tie]))
    assert r.stats().stack_overflows == 0
    r.close()


@pytest.mark.parametrize("n", [2, 3, 64, 3000])
def test_coincident_triangles_build_a_tree(n):
    print(f"case: {n} equal triangles", flush=True)
    rng = np.random.default_rng(n)
    s = _scene(n, rng, same=True)
    r = P.Renderer(8, 8)
    r.set_scene(s)
    c = s.export()["tri_pos"][0].reshape(3, 3).mean(0)
    org = rng.uniform(-4, 4, (200, 3))
    rays = np.concatenate([org, np.zeros((200, 1)), c - org, np.full((200, 1), 3e38)], 1).astype(np.float32)
    t, _, _, prim = r.intersect(rays)
    assert (prim != P.MISS).all() and np.allclose(t, 1.0, atol=1e-4)
    r.close()


def test_emitters_and_normals_keep_input_order():
    """Per path against the oracle: many emitters of both kinds scattered over the input, half of
    the triangles with normals of their own, then an emission edit each way."""
    print("case: emitters and normals", flush=True)
    rng = np.random.default_rng(5)
    n = 700
    s = P.Scene()
    mats = [s.add_material(P.LAMBERTIAN, (0.6, 0.5, 0.4), (3, 2, 1) if k == 3 else (0, 0, 0)) for k in range(6)]
    pos = np.asarray(_scene(n, rng).export()["tri_pos"]).reshape(n, 9)
    v = pos.reshape(n, 3, 3)
    g = np.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    g /= np.linalg.norm(g, axis=1, keepdims=True)
    nrm = np.repeat(g[:, None, :], 3, 1)
    nrm[::2] += 0.2 * rng.normal(size=nrm[::2].shape)
    nrm /= np.linalg.norm(nrm, axis=2, keepdims=True)
    s.add_triangles(pos, [mats[k] for k in rng.integers(0, 6, n)], normals=nrm.reshape(n, 9))
    s.add_spheres(rng.uniform(-2, 2, (5, 3)), np.full(5, 0.2), [mats[k] for k in (3, 0, 3, 4, 1)])
    W = H = 48
    spp = 4
    r = P.Renderer(W, H)
    r.set_scene(s)
    r.set_max_depth(5)
    pix, smp = np.tile(np.arange(W * H), spp), np.repeat(np.arange(spp), W * H)
    for edit in ({}, {4: (1, 2, 3)}, {4: (0, 0, 0), 3: (0, 0, 0), 0: (2, 2, 2)}):
        a = s.export()
        for k, e in edit.items():
            r.set_material(mats[k], P.LAMBERTIAN, (0.6, 0.5, 0.4), e)
            a["mat_emit"][mats[k]] = e
        r.render(spp)
        o = O.Scene(a, W, H)
        frac, self_frac, _ = path_agreement(o, r.path_radiance(W * H * spp), pix, smp, max_depth=5)
        print(f"per path: {frac:.5f} (oracle FP32 against FP64: {self_frac:.5f})", flush=True)
        assert frac > 0.99
    r.close()
