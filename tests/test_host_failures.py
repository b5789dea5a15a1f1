"""What the renderer's host code does after a call has failed, and what it hands to kernels, on a HIP
runtime double (host/hip_double.cpp): no GPU, allocations that fail on request, launches that are
recorded and do not run."""
import os
import subprocess
import sys
import textwrap

import pytest

import pathed_capi as P

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, os, struct, sys
double = C.CDLL({double!r}, mode=C.RTLD_GLOBAL)
double.double_name.restype = C.c_char_p
double.double_room.restype = C.c_size_t
double.double_watch.argtypes = [C.c_char_p, C.c_int, C.c_size_t]
double.double_room.argtypes = [C.c_void_p]
sys.path.insert(0, {package!r})
import numpy as np
import pathed_capi as P

def watch(name, index, size):
    double.double_watch(name.encode(), index, size)
    watch.size = size

def launches():
    # (kernel, blocks, threads, the watched argument's bytes) of each watched launch so far
    out = []
    for k in range(double.double_launches()):
        grid, arg = (C.c_uint * 2)(), C.create_string_buffer(watch.size)
        double.double_grid(k, grid)
        double.double_arg(k, arg)
        out.append((double.double_name(k).decode(), grid[0], grid[1], arg.raw))
    return out

def fails(f, *args):
    try:
        f(*args)
    except P.PtError:
        return
    raise AssertionError("the call did not fail")
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("double") / "hip_double.so")
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           os.path.join(HERE, "host", "hip_double.cpp"), "-o", lib])
    prelude = PRELUDE.format(double=lib, package=os.path.dirname(P.__file__))

    def go(body, *args):
        res = subprocess.run([sys.executable, "-c", prelude + textwrap.dedent(body), *map(str, args)], capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stdout + res.stderr

    return go


@pytest.mark.parametrize("kind", [P.RENDERER_OPTIX, P.RENDERER_GUIDED])
def test_a_failed_pass_keeps_the_reset_pending(run, kind):
    """A new image's first pass fails for want of memory; the next one still starts from empty sums
    (k_accumulate's PassEnd::fresh, its last argument's first member)."""
    run("""
    s = P.Scene.preset(0)
    failed = 0
    for n in range(1, 100):
        r = P.Renderer(8, 8)
        r.set_type(int(sys.argv[1]))
        r.set_scene(s)
        watch("12k_accumulateE", 6, 4)
        r.render(1)
        r.reset()
        double.double_fail_at(n)
        try:
            r.render(100000)   # the path pool grows
            break
        except P.PtError:
            failed += 1
        double.double_fail_at(0)
        assert r.spp() == 0
        r.set_option(P.OPT_POOL_PATHS, 4096)
        r.render(1)
        fresh = [struct.unpack("i", a)[0] for _, _, _, a in launches()]
        assert fresh == [0, 1], (n, fresh)   # loading the scene cleared the sums for the first
        assert r.spp() == 1
    assert failed >= 13, failed
    """, kind)


def test_a_pool_that_could_not_grow_is_allocated_again(run):
    """The path pool fails to grow at each of its arrays in turn; the next pass, which the old capacity
    would hold, gets arrays that exist and hold its queues (k_shade's path state, arguments 4 to 16)."""
    run("""
    s = P.Scene.preset(0)
    for n in range(1, 14):
        r = P.Renderer(8, 8)
        r.set_scene(s)
        r.set_option(P.OPT_PROFILE_KERNELS, 1)
        r.render(1)
        double.double_fail_at(n)
        fails(r.render, 100000)
        double.double_fail_at(0)
        for arg in range(4, 17):
            watch("7k_shade", arg, 8)
            r.render(1)
            assert launches()
            for _, _, _, a in launches():
                assert double.double_room(struct.unpack("P", a)[0]) >= 64 * 64 * 16, (n, arg)
    """)


def test_guiding_memory_that_could_not_grow_is_allocated_again(run):
    """The same for the arrays of a guided pass: the mixtures, features, training records and record
    indices of the next pass (k_shade's GuideShadeArgs, argument 17)."""
    run("""
    s = P.Scene.preset(0)
    for n in range(14, 19):   # after the pool's thirteen
        r = P.Renderer(8, 8)
        r.set_type(P.RENDERER_GUIDED)
        r.set_option(P.OPT_GUIDE_TRAIN_STEPS, 0)
        r.set_scene(s)
        r.render(1)
        double.double_fail_at(n)
        fails(r.render, 100000)
        double.double_fail_at(0)
        watch("7k_shade", 17, 56)
        r.render(1)
        mix, feat, records, seg, rec_in, rec_out, _ = struct.unpack("PPPi4xPPf4x", launches()[0][3])   # a guided bounce
        assert seg > 0 and double.double_room(records) >= 64 * seg * 64, n
        for p, size in ((mix, 64), (feat, 32), (rec_in, 4), (rec_out, 4)):
            assert double.double_room(p) >= 64 * 64 * size, (n, size)
    """)


def test_a_scene_that_could_not_be_loaded_leaves_no_freed_memory_in_use(run):
    """A scene load fails at each of its allocations in turn: the renderer then has no scene, and says so,
    until one is loaded; what it does with that, it does with memory that is there."""
    run("""
    def scene(n):
        s = P.Scene()
        m = s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
        e = s.add_material(P.LAMBERTIAN, (0, 0, 0), (1, 1, 1))
        for _ in range(100 * n):
            s.add_material(P.MIRROR, (1, 1, 1))   # no array of the old scene's size fits the new one's
        tri = np.arange(9 * n, dtype=np.float32).reshape(n, 9) % 7
        s.add_triangles(tri, np.arange(n) % 2, normals=np.ones((n, 9), np.float32))
        s.set_environment(np.ones((4, 8, 4), np.float32))
        return s

    old, new = scene(1), scene(2)   # (trees of one node, which need no kernel to be built)
    for n in range(1, 100):
        r = P.Renderer(8, 8)
        r.set_scene(old)
        r.render(1)
        double.double_fail_at(n)
        try:
            r.set_scene(new)
            break
        except P.PtError:
            pass
        double.double_fail_at(0)
        edit = lambda: r.set_material(1, P.LAMBERTIAN, emit=(2, 2, 2))
        for call in (lambda: r.render(1), edit, lambda: r.hit_test(1, 1), lambda: r.intersect(np.ones((1, 8), np.float32)), lambda: r.autotune(1)):
            try:
                call()
            except P.PtError as e:
                assert "no scene" in str(e), (n, e)
            else:
                raise AssertionError("a call went on without a scene")
        r.set_scene(old)
        for kernel, index, call in [("k_paths", 0, lambda: r.render(1))] + [("k_emitters_small", k, edit) for k in (1, 2, 3, 4, 10)]:
            size = 40 if kernel == "k_paths" else 8
            watch("%d%s" % (len(kernel), kernel), index, size)
            call()
            for p in struct.unpack("%dP" % (size // 8), launches()[-1][3]):
                assert double.double_room(p) > 0, (n, kernel, index)
    assert n > 10, n
    """)


@pytest.mark.parametrize("empty", [(0,), (1,), (2,), (0, 2), (0, 1, 2)])
def test_a_batch_render_without_primitives_has_a_node_of_its_own(run, empty):
    """Renders of an environment alone in a batch: their rays start at a node of theirs, inside the merged
    array, that has no children (k_extend's scene view, k_raygen_batch's chunk)."""
    run("""
    empty = [int(a) for a in sys.argv[1:]]
    b = P.Batch()
    for k in range(3):
        s = P.Scene()
        m = s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
        if k not in empty:
            s.add_triangles([[0, 0, 0, 1, 0, 0, 0, 1, 0]], [m])
        s.set_environment(np.ones((2, 4, 4), np.float32))
        b.add(s, 8, 8, 1, 2)
    b.set_option(P.OPT_BATCH_GRAPH, 0)
    watch("8k_extend", 0, 56)
    b.run()
    nodes, n_nodes = struct.unpack("5P4i", launches()[0][3])[0:7:6]
    watch("14k_raygen_batch", 0, 96)
    b.run()
    renders = struct.unpack("12Q", launches()[0][3])[10]
    size = double.double_room(renders) // 3
    roots = [struct.unpack("i", C.string_at(renders + k * size, 4))[0] for k in range(3)]
    assert len(set(roots)) == 3 and 0 <= min(roots) and max(roots) < n_nodes and double.double_room(nodes) >= 128 * n_nodes, (roots, n_nodes)
    for k in empty:
        node = C.string_at(nodes + 128 * roots[k], 128)
        boxes = np.frombuffer(node, np.float32, 24).reshape(3, 2, 4)
        assert np.all(boxes[:, 0] == np.float32(1e30)) and np.all(boxes[:, 1] == np.float32(-1e30))   # inverted: nothing hits them
        assert struct.unpack("4i", node[96:112]) == (0x7fffffff,) * 4
    """, *empty)


@pytest.mark.parametrize("count", [2, 5])
def test_a_batch_keeps_its_renders_vertex_normals_in_threes(run, count):
    """A smooth triangle's tag counts triples of normals: what a batch adds to it (k_rebase_prims's offset)
    counts triples too, and each render's first triple lies inside the merged array (k_extend's scene view)."""
    run("""
    count = int(sys.argv[1])
    b = P.Batch()
    for k in range(count):
        s = P.Scene()
        s.add_triangles([[0, 0, 0, 1, 0, 0, 0, 1, 0]], [s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))])
        s.set_environment(np.ones((2, 4, 4), np.float32))
        b.add(s, 8, 8, 1, 2)
    b.set_option(P.OPT_BATCH_GRAPH, 0)
    watch("14k_rebase_prims", 3, 4)
    b.run()
    offsets = [struct.unpack("i", l[3])[0] for l in launches()]
    assert len(offsets) == count and offsets == sorted(set(offsets)) and offsets[0] == 0, offsets
    watch("8k_extend", 0, 56)
    b.run()
    normals = struct.unpack("5P", launches()[0][3][:40])[2]
    assert double.double_room(normals) >= 16 * 3 * (offsets[-1] + 1), (offsets, double.double_room(normals))
    """, count)


@pytest.mark.parametrize("width,height", [(1, 1), (1 << 28, 1), (1, 1 << 28), (1 << 14, 1 << 14)])
def test_the_normals_view_of_the_largest_images_has_a_grid(run, width, height):
    run("""
    r = P.Renderer(int(sys.argv[1]), int(sys.argv[2]))
    r.set_scene(P.Scene.preset(0))
    r.set_type(P.RENDERER_NORMALS)
    watch("9k_normals", 0, 8)
    r.render(1)
    (name, blocks, threads, _), = launches()
    assert 1 <= blocks <= 11 * 256 and threads == 128, blocks
    assert int(sys.argv[1]) * int(sys.argv[2]) == 1 or blocks == 11 * 256
    """, width, height)


def test_the_normals_view_leaves_the_pool_option(run):
    run("""
    r = P.Renderer(128, 96)
    r.set_scene(P.Scene.preset(0))
    r.set_option(P.OPT_POOL_PATHS, 4096)
    r.set_type(P.RENDERER_NORMALS)
    r.render(1)
    assert r.get_option(P.OPT_POOL_PATHS) == 4096
    r.set_type(P.RENDERER_OPTIX)
    watch("12k_accumulateE", 0, 4)
    r.render(1)
    assert len(launches()) == 3   # chunks of 4096 paths
    """)


def test_images_are_read_from_any_thread_and_device(run):
    """A renderer of one device read while another is current, and from a thread that never chose one: the
    events of the copy are of the stream's device, and the caller's device stays what it was."""
    run("""
    import threading
    double.double_devices(2)
    current = C.c_int()
    for own, other in ((0, 1), (1, 0)):
        assert double.hipSetDevice(own) == 0
        r = P.Renderer(40, 30)
        r.set_scene(P.Scene.preset(0))
        r.render(1)
        assert double.hipSetDevice(other) == 0
        for read in (r.radiance, r.radiance_sum, r.rgba8):
            read()
            double.hipGetDevice(C.byref(current))
            assert current.value == other
        read = []
        t = threading.Thread(target=lambda: read.append(r.radiance()))
        t.start()
        t.join()
        assert len(read) == 1
    """)


@pytest.mark.parametrize("lds,nee,blocks", [(16, 1, 8), (16, 0, 8), (32, 1, 6), (32, 0, 8)])
def test_whole_path_grids_are_what_fits_the_chip(run, lds, nee, blocks):
    """Blocks of k_paths per CU by their LDS (160 KB; 11 KB of 16 stack rows, 19 KB of 32, 5.5 KB of shadow
    lists) and registers: a second go of a few blocks takes as long as the first."""
    run("""
    lds, nee, blocks = (int(a) for a in sys.argv[1:])
    r = P.Renderer(1024, 1024)
    r.set_scene(P.Scene.preset(0))
    r.set_option(P.OPT_TRACE_LDS_STACK, lds)
    r.set_nee(nee)
    watch("7k_paths", 3, 4)
    r.render(1)
    (_, grid, threads, _), = launches()
    assert grid == 256 * blocks and threads == 128, grid
    """, lds, nee, blocks)


def test_whole_paths_up_to_the_limit(run):
    run("""
    s = P.Scene()
    s.add_triangles([[0, 0, 0, 1, 0, 0, 0, 1, 0]], [s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))])   # one node
    for height, whole in ((2048, 1), (2049, 0)):
        r = P.Renderer(4096, height)
        r.set_scene(s)
        watch("7k_paths", 3, 4)
        r.render(1)
        assert len(launches()) == whole
    """)


def test_the_autotuner_tries_no_more_trace_blocks_than_a_cu_holds(run):
    """160 KB of LDS a CU, 14.5 KB a block of the queue traversal: eleven."""
    run("""
    r = P.Renderer(64, 64)
    r.set_scene(P.Scene.preset(0))
    r.set_type(P.RENDERER_GUIDED)   # always through the queues
    r.set_option(P.OPT_GUIDE_TRAIN_STEPS, 0)
    watch("7k_trace", 0, 8)
    r.autotune(2)
    grids = {g for _, g, _, _ in launches()}
    assert grids and max(grids) <= 11 * 256, grids
    """)


def test_rays_that_can_hit_nothing_are_sent_as_empty_intervals(run):
    """Ray queries with undefined components, an origin that is not finite or a direction infinite on all
    axes: the slab test would accept every box for them, those of a node's unused children too.  What is
    sent to k_extend and k_shadow (arguments 4 and 5, where a ray's origin and direction are) has none."""
    run("""
    s = P.Scene()
    s.add_triangles([[0, 0, 0, 1, 0, 0, 0, 1, 0]], [s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))])
    r = P.Renderer(8, 8)
    r.set_scene(s)
    inf, nan = np.inf, np.nan
    plain = [1, 2, 3, 0.5, 0, -1, 0.25, 7]
    empty = [[nan] * 3 + plain[3:], [nan] * 3 + [-inf, 0, 0, 1, inf], [inf] + plain[1:], [0, -inf] + plain[2:], [nan] + plain[1:], plain[:3] + [nan] + plain[4:],
             plain[:7] + [nan], plain[:4] + [nan, 0, 1, 7], plain[:4] + [inf, -inf, inf, 7], [nan, nan, 1e30, nan, 0, 0, 0, inf], [nan] * 8, [inf] * 8]
    kept = [plain, plain[:4] + [0, 0, 0, 7], plain[:4] + [inf, 0, 1, 7], [1e30, 1e30, 1e30] + plain[3:], [3e38] * 3 + plain[3:], [0.] * 8, plain[:4] + [3e38] * 4]
    bounds = [plain[:3] + [-inf] + plain[4:7] + [inf], plain[:3] + [inf] + plain[4:7] + [-inf]]
    big = np.finfo(np.float32).max
    rays = np.array(empty + kept + bounds, np.float32)
    want = np.array([[0, 0, 0, big, 0, 0, 1, -big]] * len(empty) + kept + [plain[:3] + [-big] + plain[4:7] + [big], plain[:3] + [inf] + plain[4:7] + [-inf]], np.float32)
    for any_hit, kernel in ((0, "8k_extend"), (1, "8k_shadow")):
        sent = []
        for arg in (4, 5):
            watch(kernel, arg, 8)
            r.intersect(rays, any_hit=bool(any_hit))
            (_, _, _, p), = launches()
            sent.append(np.frombuffer(C.string_at(struct.unpack("P", p)[0], 16 * len(rays)), np.float32).reshape(-1, 4))
        o, d = sent
        assert np.array_equal(o[:, :3], want[:, :3]) and np.array_equal(d[:, :3], want[:, 4:7]), (o, d)
        if any_hit:
            assert np.array_equal(o[:, 3], want[:, 7])
        else:
            assert np.array_equal(o[:, 3], want[:, 3]) and np.array_equal(d[:, 3], want[:, 7]), (o, d)
    """)


def test_ray_queries_of_a_scene_without_primitives_launch_nothing(run):
    """Every ray misses.  (The kernels' way without nodes takes extension rays only: a shadow ray's end is
    written to the path that its load has noted, and nothing is loaded there.)"""
    run("""
    s = P.Scene()
    s.add_material(P.LAMBERTIAN, (0.5, 0.5, 0.5))
    r = P.Renderer(8, 8)
    r.set_scene(s)
    for kernel in ("8k_shadow", "8k_extend"):
        watch(kernel, 0, 8)
        for any_hit in (False, True):
            t, u, v, prim = r.intersect(np.ones((70, 8), np.float32), any_hit=any_hit)
            assert np.all(t == -1) and not u.any() and not v.any() and np.all(prim == P.MISS)
        assert not launches()
    """)
