"""Performance cases of the path tracer: what its users have it do, from one click to a 64-sample still.

Every case goes through the ctypes binding (pathed_capi) as a program would call it.  Sizes are those of
bench.py (icosphere of 1,310,720 triangles at 1024x1024 and 64 samples, room of 4,000,032 triangles at
2048x1024, batches of geodesic spheres), of the tests (Cornell box at 256x256) and generic ones.  Images are
functions of the scene, the camera and the PCG32 seed, all of which come from the case's seed; a render
starts from an empty accumulator, so a pass can be repeated.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-pathed_amd"))
import pathed_capi as P  # noqa: E402

ICOSPHERE_8 = 1310720  # triangles of the subdivision-8 icosphere
ROOM = 4000032


def listed():
    return [
        # a click in the viewport: the material under one pixel
        dict(name="pick", kind="pick", scene="geodesic", tris=100000, width=512, height=512),
        # the environment's sampling tables rebuilt from a map in device memory
        dict(name="env_tables", kind="env", width=1024, height=512, sin_theta=False),
        # dragging the camera of the default scene: one sample per pixel, framebuffer bytes on the host
        dict(name="drag_cornell", kind="drag", scene="cornell", tris=12, width=256, height=256, depth=5),
        # the default scene as a small still, no next-event estimation (the naive estimator)
        dict(name="cornell_naive", kind="still", scene="cornell", tris=12, width=333, height=251, spp=4, depth=5, nee=False, consistent=False),
        # the default scene as a small still
        dict(name="cornell", kind="still", scene="cornell", tris=12, width=256, height=256, spp=16, depth=6, nee=True, consistent=False),
        # the shading-normal view of a mesh
        dict(name="normals", kind="normals", scene="geodesic", tris=327680, width=1280, height=720),
        # a progressive pass of a mesh under an environment, an odd window size
        dict(name="preview", kind="still", scene="geodesic", tris=327680, width=641, height=359, spp=1, depth=8, nee=True, consistent=False),
        # a mesh with a material per face loaded into the renderer, and its first image
        dict(name="load", kind="load", scene="geodesic", tris=ICOSPHERE_8, width=256, height=256, spp=1, depth=8, nee=True),
        # a dozen thumbnails of different meshes as one batch
        dict(name="batch", kind="batch", renders=12, res=512, spp=16, tris=200000),
        # a progressive pass of the learned-guiding renderer from a fresh network, its training steps included
        dict(name="guided_room", kind="guided", scene="room", tris=1000000, width=1024, height=512, spp=1, depth=16),
        # a progressive pass of a large interior
        dict(name="room", kind="still", scene="room", tris=ROOM, width=2048, height=1024, spp=1, depth=16, nee=True, consistent=True),
        # a finished still of a large mesh
        dict(name="icosphere", kind="still", scene="geodesic", tris=ICOSPHERE_8, width=1024, height=1024, spp=64, depth=8, nee=True,
             consistent=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick", "env", "drag", "still", "still", "still", "normals", "load", "batch", "guided"])
    if kind == "env":
        w = _log(rng, 64, 2048)
        return dict(kind=kind, width=w, height=max(2, w // 2 + rng.choice([0, 0, -1, 3])), sin_theta=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind=kind, renders=_log(rng, 2, 16), res=_log(rng, 128, 512), spp=_log(rng, 4, 16), tris=_log(rng, 10000, 200000))
    scene = "room" if kind == "guided" else "geodesic" if kind in ("pick", "normals", "load") else rng.choice(["cornell", "geodesic", "room"])
    c = dict(kind=kind, scene=scene)
    c["tris"] = 12 if scene == "cornell" else _log(rng, 100000, 2000000) if scene == "room" else _log(rng, 2000, ICOSPHERE_8)
    c["width"] = _log(rng, 96, 1536)
    c["height"] = max(16, int(c["width"] * rng.uniform(0.5, 1.0)))
    if kind in ("pick", "normals"):
        return c
    c["depth"] = rng.randint(3, 16 if scene == "room" else 8)
    if kind == "drag":
        c["width"], c["height"] = min(c["width"], 720), min(c["height"], 720)
        return c
    if kind in ("guided", "load"):
        c["width"], c["height"], c["spp"] = min(c["width"], 1024), min(c["height"], 512), 1
        if kind == "load":
            c["nee"] = True
        return c
    most = (1 << 22 if scene == "room" else 1 << 25) // (c["width"] * c["height"])
    c["spp"] = _log(rng, 1, max(1, min(64, most)))
    c["nee"] = rng.random() < 0.8
    c["consistent"] = rng.random() < 0.3
    return c


# ---------------------------------------------------------------------------------------------


def _scene(case, seed):
    if case["scene"] == "cornell":
        return P.Scene.preset(0)
    return P.Scene.preset(2 if case["scene"] == "room" else 4, seed=seed % 1000003, param=case["tris"])


def _camera(case, rng):
    """A camera beside the scene's own one: (origin, target, up, vfov, flip)."""
    if case["scene"] == "cornell":
        o, t, fov = (0.0, 1.0, 6.8), (0.0, 1.0, 0.0), 19.5
    elif case["scene"] == "room":
        o, t, fov = (-2.4, 1.4, 2.6), (0.5, 1.1, -1.0), 55.0
    else:
        o, t, fov = (0.0, 0.35, 3.2), (0.0, 0.0, 0.0), 40.0
    o = tuple(x + d for x, d in zip(o, rng.uniform(-0.05, 0.05, 3)))
    return o, t, (0.0, 1.0, 0.0), fov / 180.0 * math.pi, False


def _env_map(case, seed):
    """A sky: log-normal texels and one small bright sun."""
    rng = np.random.default_rng(seed)
    w, h = case["width"], case["height"]
    m = np.ones((h, w, 4), np.float32)
    m[..., :3] = np.exp(rng.standard_normal((h, w, 1)))
    m[int(rng.integers(0, h)), int(rng.integers(0, w)), :3] = 1e4
    return m


def _thumbnail(case, i):
    """Side and samples of a batch's render i: the case's, halves and quarters of them, in all pairs."""
    return case["res"] >> (i % 3), max(1, case["spp"] >> (i // 3 % 3))


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "env":
        w, h = case["width"], case["height"]
        dev = dict(dtype=torch.float32, device="cuda")
        return dict(case=case, rgba=torch.from_numpy(_env_map(case, seed)).cuda(), rows=torch.empty((h, w, 2), **dev),
                    marginal=torch.empty((h, 2), **dev), pdf=torch.empty((h, w), **dev))
    if kind == "batch":
        b = P.Batch()
        for i in range(case["renders"]):
            res, spp = _thumbnail(case, i)
            b.add(P.Scene.preset(4, seed=int(rng.integers(1, 1 << 30)), param=_log_np(rng, 10000, case["tris"])), res, res, spp, 8)
        return dict(case=case, batch=b)
    scene = _scene(case, seed)
    r = P.Renderer(case["width"], case["height"])
    r.set_seed(seed)
    st = dict(case=case, r=r, scene=scene, camera=_camera(case, rng))
    if kind != "load":
        r.set_scene(scene)
        r.set_camera(*st["camera"])
    if kind == "pick":
        # a pixel of the middle of the window, where the mesh is
        st["at"] = tuple(int(s * (0.5 + 0.2 * u)) for s, u in zip((case["width"], case["height"]), rng.uniform(-1, 1, 2)))
    elif kind == "normals":
        r.set_type(P.RENDERER_NORMALS)
    else:
        r.set_max_depth(case["depth"])
        r.set_nee(case.get("nee", True))
        if kind == "guided":
            r.set_type(P.RENDERER_GUIDED)
        if case.get("consistent") or kind == "guided":
            r.set_option(P.OPT_CONSISTENT_MIS, 1)
    return st


def _log_np(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(max(lo, hi))))))


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "env":
        P.check(P.lib().pt_env_tables_noalloc(st["rgba"].data_ptr(), case["width"], case["height"], int(case["sin_theta"]), st["rows"].data_ptr(),
                                              st["marginal"].data_ptr(), st["pdf"].data_ptr(), torch.cuda.current_stream().cuda_stream))
        # table entries are (probability, alias index bits)
        return dict(rows=st["rows"].view(torch.int32), marginal=st["marginal"].view(torch.int32), texel_pdf=st["pdf"])
    if kind == "batch":
        b = st["batch"]
        b.run()
        return [b.radiance(i) for i in range(case["renders"])]
    r = st["r"]
    if kind == "pick":
        material, hit = r.hit_test(*st["at"])
        return dict(material=material, hit=hit)
    if kind == "load":
        r.set_scene(st["scene"])
        r.set_camera(*st["camera"])
        r.render(case["spp"])
        return r.radiance()
    if kind == "drag":
        r.set_camera(*st["camera"])
        r.render(1)
        return r.rgba8()
    if kind == "guided":
        r.set_option(P.OPT_GUIDE_RESET, 1)
    r.reset()
    r.render(case.get("spp", 1))
    return r.radiance()


# Rays a camera path leads to, itself included (continuation and shadow rays), as bench.py's stats give them
RAYS = {"cornell": 6.0, "geodesic": 1.9, "room": 15.0}


def work(case):
    """Scene arrays read once, outputs written once; of arithmetic, per ray one root-to-leaf descent of a
    4-wide tree (4 slab tests of 18 operations a level), a leaf's triangle test (60) and one shaded vertex
    (400).  The trees' inner nodes are the renderer's own, so they count as arithmetic only."""
    kind = case["kind"]
    if kind == "env":
        n = case["width"] * case["height"]
        return {"bytes": n * (16 + 8 + 4) + case["height"] * 8, "flops": n * 8}

    def rays(n, tris):
        return n * (max(1.0, math.log(max(tris, 2), 4)) * 72 + 460)

    if kind == "batch":
        # the middle of the range of triangles, which is drawn on a log scale
        n, tris = case["renders"], int(math.sqrt(10000 * max(10000, case["tris"])))
        shapes = [_thumbnail(case, i) for i in range(n)]
        return {"bytes": n * (tris * 80 + 1024 * 512 * 28) + sum(a * a * 12 for a, _ in shapes),
                "flops": rays(sum(a * a * s for a, s in shapes) * RAYS["geodesic"], tris)}
    tris, pix = case["tris"], case["width"] * case["height"]
    if kind == "pick":
        return {"bytes": 24 * 48, "flops": rays(1, tris)}
    scene = tris * (48 + (32 if case["scene"] == "geodesic" else 0)) + {"cornell": 0, "geodesic": 1024 * 512 * 28, "room": 2048 * 1024 * 28}[case["scene"]]
    if kind == "normals":
        # one centre ray per pixel and at most one primitive record each
        return {"bytes": min(pix, tris) * 48 + pix * 12, "flops": rays(pix, tris)}
    paths = pix * case.get("spp", 1)
    w = {"bytes": min(paths * 2 * 80, scene) + pix * (4 if kind == "drag" else 12), "flops": rays(paths * RAYS[case["scene"]], tris)}
    if kind == "load":
        w["bytes"] += 2 * scene
    if kind == "guided":
        # the network at about 6 guided vertices a path, then 16 training steps of 2^18 records (forward
        # and twice that backward)
        layer = 2 * 5 * 64 * 64
        w["flops"] += paths * 6 * layer + 16 * (1 << 18) * 3 * layer
    return w


def exact(case, seed):
    """The environment's texel densities in 64 bits.  An image is a function of FP32 random walks (a last-bit
    difference sends a path elsewhere), and picks and table entries are whole numbers: they have no such value."""
    if case["kind"] != "env":
        return None
    m = _env_map(case, seed).astype(np.float64)
    w, h = case["width"], case["height"]
    wts = m[..., :3].sum(-1)
    if case["sin_theta"]:
        wts = wts * np.sin((np.arange(h) + 0.5) / h * math.pi)[:, None]
    return dict(rows=None, marginal=None, texel_pdf=wts / wts.sum() * (w * h) / (2.0 * math.pi**2))
