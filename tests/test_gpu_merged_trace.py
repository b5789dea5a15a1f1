"""A bounce's shadow rays traced in one launch with the next bounce's extension rays against the two
launches (which run while kernels are timed): the same images bit for bit and the same ray counts, from
one path to several chunks, at depths with no, one and many such launches, with deep stacks that spill,
and in a batch."""
import numpy as np
import pytest

import pathed_capi as P

pytestmark = pytest.mark.gpu


def _image(scene, W, H, spp, depth, pool, lds, profile):
    r = P.Renderer(W, H)
    r.set_type(P.RENDERER_GUIDED)   # always traced through the queues
    r.set_option(P.OPT_GUIDE_TRAIN_STEPS, 0)
    r.set_option(P.OPT_TRACE_LDS_STACK, lds)
    if pool:
        r.set_option(P.OPT_POOL_PATHS, pool)
    r.set_scene(scene)
    r.set_max_depth(depth)
    r.set_option(P.OPT_PROFILE_KERNELS, profile)
    r.render(spp)
    st = r.stats()
    out = [r.radiance_sum(), np.array(st.bounce_rays), np.array(st.bounce_shadow), st.extension_rays, st.shadow_rays]
    assert st.stack_overflows == 0
    r.close()
    return out


@pytest.mark.parametrize("W,H,spp,depth,pool", [(1, 1, 1, 2, 0), (63, 1, 1, 3, 0), (65, 1, 1, 1, 0), (33, 7, 3, 9, 0), (150, 90, 2, 4, 4096),
                                                (641, 359, 2, 16, 0)])
@pytest.mark.parametrize("kind", [0, 2, 4])
def test_merged_trace_equals_two_launches(kind, W, H, spp, depth, pool):
    print(f"case: preset {kind} {W}x{H}, {spp} spp, depth {depth}, pool {pool}", flush=True)
    scene = P.Scene.preset(kind, 3, 100000 if kind else 0)
    for lds in (16, 32):
        for k, (a, b) in enumerate(zip(_image(scene, W, H, spp, depth, pool, lds, 0), _image(scene, W, H, spp, depth, pool, lds, 1))):
            assert np.array_equal(a, b), (lds, k)


def test_merged_trace_in_a_batch():
    jobs = [(4, 1, 12000, 256, 128, 6, 5), (2, 2, 100000, 128, 96, 3, 9), (0, 0, 0, 64, 64, 8, 6)]
    b = P.Batch()
    ref = []
    for p, s, q, w, h, spp, depth in jobs:
        sc = P.Scene.preset(p, s, q)
        b.add(sc, w, h, spp, depth)
        r = P.Renderer(w, h)
        r.set_scene(sc)
        r.set_max_depth(depth)
        r.render(spp)
        ref.append(r.radiance())
        r.close()
    for _ in range(3):
        b.run()
        for i, want in enumerate(ref):
            assert np.array_equal(b.radiance(i), want), i
    b.close()


def test_merged_trace_of_a_plain_pass_too_large_to_trace_whole():
    scene = P.Scene.preset(4, 3, 100000)
    out = []
    for profile in (0, 1):
        r = P.Renderer(1536, 1400)
        r.set_scene(scene)
        r.set_max_depth(4)
        r.set_option(P.OPT_PROFILE_KERNELS, profile)
        r.render(1)
        st = r.stats()
        out.append([r.radiance_sum(), np.array(st.bounce_rays), np.array(st.bounce_shadow)])
        assert st.bvh_nodes > 4096 and st.stack_overflows == 0
        r.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
