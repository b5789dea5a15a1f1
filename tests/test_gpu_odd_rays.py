"""Ray queries whose bounds are infinite.  (Rays that can hit nothing, from nowhere or along nothing, are
answered by an empty interval: tests/test_host_failures.py looks at what is sent for them.)"""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 5, 90, 3000])
@pytest.mark.parametrize("lds", [16, 32])
def test_infinite_bounds(n, lds):
    print(f"case: {n} triangles, {lds} stack rows", flush=True)
    rng = np.random.default_rng(n)
    c = rng.uniform(-2, 2, (n, 1, 3))
    s = P.Scene()
    s.add_triangles((c + rng.normal(size=(n, 3, 3)) * 0.4).reshape(n, 9), np.full(n, s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))))
    r = P.Renderer(8, 8)
    r.set_option(P.OPT_TRACE_LDS_STACK, lds)
    r.set_scene(s)
    k = 2000
    rays = np.zeros((k, 8), np.float32)
    rays[:, :3] = rng.uniform(-4, 4, (k, 3))
    rays[:, 4:7] = c[rng.integers(0, n, k), 0] - rays[:, :3]
    rays[:, 3], rays[:, 7] = -3e38, 3e38
    want = r.intersect(rays)
    assert (want[3] != P.MISS).any()
    inf = np.float32(np.inf)
    for tmin, tmax in ((-inf, 3e38), (-3e38, inf), (-inf, inf)):
        odd = rays.copy()
        odd[:, 3], odd[:, 7] = tmin, tmax
        for a, b in zip(r.intersect(odd), want):
            assert np.array_equal(a, b)
    odd[:, 3], odd[:, 7] = 1, -1
    assert np.all(r.intersect(odd)[3] == P.MISS) and np.all(r.intersect(odd, any_hit=True)[3] == P.MISS)
    assert r.stats().stack_overflows == 0
    r.close()
