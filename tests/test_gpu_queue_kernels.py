"""The queue kernels where an ordinary small pass no longer takes them (it is traced whole): path by path
against the oracle at awkward sizes with the kernels timed, which runs every queue kernel by itself; in passes
too large to trace whole, whose shadow and extension rays share launches; camera packets on a tree of many
levels; and the trace waves' refill threshold, on which no result depends."""
import numpy as np
import pytest

import oracle as O
import pathed_capi as P

pytestmark = pytest.mark.gpu


def _agreement(scene, W, H, spp, depth, pixels, **options):
    """Share of the pixels' paths within 1e-3 of the oracle's on the same random streams."""
    r = P.Renderer(W, H)
    r.set_scene(scene)
    r.set_max_depth(depth)
    for opt, v in options.items():
        r.set_option(getattr(P, "OPT_" + opt), v)
    r.render(spp)
    got = r.path_radiance(W * H * spp).reshape(spp, H * W, 3)[:, pixels].reshape(-1, 3)
    st = r.stats()
    r.close()
    assert st.stack_overflows == 0
    o = O.Scene(scene.export(), W, H, bvh=True)
    want = o.trace_paths(np.tile(pixels, spp), np.repeat(np.arange(spp), len(pixels)), max_depth=depth, nee=1, mode=1, tri_test=1, ref_env=0, precision=32)
    return float((np.abs(got - want).max(1) / (np.abs(want).max(1) + 1e-3) < 1e-3).mean()), st


@pytest.mark.parametrize("W,H,spp", [(1, 1, 1), (3, 5, 2), (65, 1, 3), (17, 9, 7), (130, 3, 33)])
def test_timed_queues_per_path(W, H, spp):
    print(f"case: Cornell box {W}x{H}x{spp}, kernels timed", flush=True)
    frac, st = _agreement(P.Scene.preset(0), W, H, spp, 5, np.arange(W * H), PROFILE_KERNELS=1)
    assert frac >= 0.998 if W * H * spp >= 1000 else frac == 1.0   # as through whole paths
    assert st.rays_total >= W * H * spp


@pytest.mark.parametrize("lds", [16, 32])
def test_merged_trace_per_path(lds):
    """2^20 + 1024 paths: above what is traced whole."""
    print(f"case: icosphere 1025x1024, depth 8, {lds} stack rows", flush=True)
    pixels = np.concatenate([np.arange(1025) + 1025 * y for y in range(4, 1024, 128)])
    frac, _ = _agreement(P.Scene.preset(1, seed=3, param=5), 1025, 1024, 1, 8, pixels, TRACE_LDS_STACK=lds)
    assert frac >= 0.9995


def test_camera_packets_on_a_deep_tree_per_path():
    """81,920 triangles at 64 x 64 pixels and 64 samples: 20 primitives to a run of 64 rays, the most that
    camera packets take; timed, as an untimed pass of this size is traced whole.  And against the same
    rays traced one per lane (the counting kernels), up to ties of equal distance."""
    W, H, spp = 64, 64, 64
    s = P.Scene.preset(1, seed=0, param=6)
    assert len(s.export()["tri_pos"]) * 64 <= 20 * W * H * spp
    print("case: icosphere level 6, 64x64x64, camera packets", flush=True)
    pixels = np.concatenate([np.arange(W) + W * y for y in (7, 24, 33, 50)])
    frac, st = _agreement(s, W, H, spp, 6, pixels, PROFILE_KERNELS=1)
    assert frac >= 0.9995 and st.bvh_depth >= 8
    out = []
    for opt in (P.OPT_PROFILE_KERNELS, P.OPT_TRACE_STATS):
        r = P.Renderer(W, H)
        r.set_scene(s)
        r.set_max_depth(6)
        r.set_option(opt, 1)
        r.render(spp)
        out.append(r.path_radiance(W * H * spp))
        r.close()
    assert np.all(out[0] == out[1], axis=1).mean() >= 0.9995


@pytest.mark.parametrize("kind,W,H,spp", [(P.RENDERER_OPTIX, 1025, 1024, 1), (P.RENDERER_GUIDED, 96, 80, 3)])
def test_refill_threshold_does_not_change_images(kind, W, H, spp):
    print(f"case: refill thresholds, renderer {kind}, {W}x{H}x{spp}", flush=True)
    r = P.Renderer(W, H)
    r.set_type(kind)
    r.set_option(P.OPT_GUIDE_TRAIN_STEPS, 0)
    r.set_scene(P.Scene.preset(1, seed=3, param=5))
    r.set_max_depth(6)
    images = []
    for lanes in (0, 64, 1, 17):
        r.set_option(P.OPT_TRACE_REFILL_LANES, lanes)
        r.reset()
        r.render(spp)
        images.append(r.radiance_sum())
    assert all(np.array_equal(a, images[0]) for a in images[1:]) and images[0].any()
    assert r.stats().stack_overflows == 0
    r.close()
