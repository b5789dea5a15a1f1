"""The first 21 nodes of a tree are read from LDS by the queue kernels: closest and any hits against the
oracle over trees of one node, of fewer, as many and more nodes than that."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P

pytestmark = pytest.mark.gpu


def test_trees_around_the_nodes_in_lds():
    nodes = set()
    for n in [1, 2, 3] + list(range(60, 104, 2)) + [700]:
        print(f"case: {n} triangles", flush=True)
        rng = np.random.default_rng(n)
        c = rng.normal(size=(n, 3))
        s = P.Scene()
        m = s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
        s.add_triangles(np.concatenate([c + 0.3 * rng.normal(size=(n, 3)) for _ in range(3)], 1), np.full(n, m))
        r = P.Renderer(8, 8)
        r.set_scene(s)
        k = 1000
        org = rng.normal(size=(k, 3)) * 3
        d = c[rng.integers(0, n, k)] - org
        rays = np.concatenate([org, np.zeros((k, 1)), d, np.full((k, 1), 3e38)], 1).astype(np.float32)
        o = O.Scene(s.export(), 8, 8, bvh=True)
        gt, _, _, gp = r.intersect(rays)
        ct, _, _, cp = o.intersect(rays, tri_test=1)
        assert np.array_equal(gp, cp)
        assert np.all(np.abs(gt - ct)[gp != P.MISS] <= 1e-6 * np.abs(ct[gp != P.MISS]))
        shadow = rays.copy()
        shadow[:, 3] = 1e-4
        assert np.array_equal(r.intersect(rays, any_hit=True)[3] == P.MISS, o.intersect(shadow, tri_test=1)[3] == P.MISS)
        nodes.add(r.stats().bvh_nodes)
        r.close()
    assert 1 in nodes and max(nodes) > 22 and len(nodes & set(range(17, 26))) >= 3
