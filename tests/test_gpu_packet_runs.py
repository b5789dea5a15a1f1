"""Camera packets (the queues' first bounce, which runs while kernels are timed) against the same paths
traced one ray per lane: runs of one dominant axis and one set of direction signs, runs that mix them,
runs cut short, triangles and spheres."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("look", [(1, 0.3, 0.2), (-1, 0.2, -0.3), (0.2, 1, 0.3), (-0.3, -1, 0.2), (0.3, 0.2, 1), (-0.2, 0.3, -1), (1, 1, 1), (0, 0, 1)])
def test_packets_equal_lanes(look):
    rng = np.random.default_rng(5)
    s = P.Scene()
    m = s.add_material(P.LAMBERTIAN, (0.6, 0.5, 0.4))
    e = s.add_material(P.LAMBERTIAN, (0, 0, 0), emit=(3, 2, 1))
    c = rng.normal(size=(400, 3)) * 3
    tri = np.concatenate([c + 0.6 * rng.normal(size=(400, 3)) for _ in range(3)], 1)
    s.add_triangles(tri, np.where(np.arange(400) % 7 == 0, e, m))
    s.add_spheres(rng.normal(size=(40, 3)) * 3, np.full(40, 0.3), np.full(40, m))
    for W, H, spp in ((33, 21, 16), (13, 11, 37)):
        print(f"case: look {look}, {W}x{H}, {spp} spp", flush=True)
        s.set_camera([0.1, 0.2, 0.05], np.add([0.1, 0.2, 0.05], look), [0.1, 0.9, 0.4], 1.2)
        out = []
        for profile in (0, 1):
            r = P.Renderer(W, H)
            r.set_scene(s)
            r.set_max_depth(3)
            r.set_option(P.OPT_PROFILE_KERNELS, profile)
            r.render(spp)
            out.append((r.radiance_sum(), r.stats().extension_rays))
            r.close()
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1] and out[0][0].any()
