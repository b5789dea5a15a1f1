"""A tree of thousands of 4-wide levels: concentric spheres, of which the PLOC builder merges one pair a
step (every sphere's best partner is the smallest there is), so that its binary tree is a chain and the
4-wide one a third as deep.  The same image and picks as from the LBVH, whose tree is shallow."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3000, 13000])
def test_concentric_spheres(n):
    print(f"case: {n} concentric spheres", flush=True)
    s = P.Scene()
    mats = [s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5)) for _ in range(4)]
    s.add_spheres(np.zeros((n, 3)), 1 + np.arange(n) / 16384, [mats[k % 4] for k in range(n)])
    s.set_camera([0, 0, 5], [0, 0, 0], [0, 1, 0], 0.9)
    out = []
    for builder in (P.BVH_LBVH, P.BVH_PLOC):
        r = P.Renderer(24, 16)
        r.set_option(P.OPT_BVH_BUILDER, builder)
        r.set_scene(s)
        r.set_type(P.RENDERER_NORMALS)
        r.render(1)
        st = r.stats()
        print(f"  builder {builder}: {st.bvh_depth} levels, {st.bvh_nodes} nodes", flush=True)
        out.append((r.radiance_sum(), [r.hit_test(x, 8) for x in range(0, 24, 3)]))
        assert st.stack_overflows == 0 and (builder == P.BVH_LBVH or st.bvh_depth >= n // 3)
        r.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    assert out[0][1][4] == (mats[(n - 1) % 4], True)
