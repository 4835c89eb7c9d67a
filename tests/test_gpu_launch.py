"""Launch shapes of the render kernels (wave_item, split_tile, draw_form):
tile counts around a workgroup, around a round of workgroups over the XCDs and
on either side of 16384 tiles, one wave a workgroup (byte offsets) and four
(word indices), as a plain draw, a hardware-scheduled launch of views and a
persistent one.  Pictures against the oracle's, ray and step totals against the
oracle's and each other's."""
import ctypes as C
import math

import numpy as np
import pytest

from test_gpu_parity import RGB_TOL

pytestmark = pytest.mark.gpu

GRIDS = [(24, 20, 40), (4096, 600, 2)]  # byte offsets; 4 X Y >= 2^23: word indices


def tiles(size):
    return -(-size[0] // 8) * -(-size[1] // 8)


SMALL = [(1, 1), (9, 3), (23, 8), (245, 5), (256, 8), (257, 8), (17, 83), (72, 50), (61, 64), (33, 99), (3, 1030)]
LARGE = [(1024, 1024), (1025, 1021)]


def test_sizes_lie_on_the_edges():
    assert [tiles(s) for s in SMALL] == [1, 2, 3, 31, 32, 33, 33, 63, 64, 65, 129]
    assert [tiles(s) for s in LARGE] == [16384, 16512]


@pytest.fixture(scope="module", params=GRIDS, ids=["byte_offset32", "index32"])
def scene(gpu, request):
    """Cells that are empty, jump or solid at random: the walks of one wave
    differ in length."""
    dims = request.param
    rng = np.random.default_rng(17)
    cells = dims[0] * dims[1] * dims[2]
    world = np.full(cells, -1, np.int32)
    jump = rng.random(cells) < 0.3
    world[jump] = (-rng.uniform(0.5, 3.0, int(jump.sum())).astype(np.float32)).view(np.int32)
    solid = rng.random(cells) < 0.03
    world[solid] = rng.integers(0, 1 << 24, int(solid.sum()))
    ctx = gpu.Context(dims)
    ctx.upload(world)
    yield dims, world, ctx
    ctx.close()


def frame(gpu, dims, size):
    f = gpu.frame_defaults(dims[0], *size)
    f.cam_pos[:] = [0.4 * dims[0], 0.55 * dims[1], 0.6 * dims[2]]
    f.rotate_matrix[:] = gpu.camera_matrix(0.1, 0.5 * math.pi - 0.05).tolist()  # along x, which both grids have
    f.aspect_ratio = size[0] / size[1]
    for i in range(6):  # a group of four lights and a part of one
        L = f.lights[i]
        L.pos[:] = [f.cam_pos[0] + 3.0 * i, f.cam_pos[1] + 1.0, f.cam_pos[2]]
        L.rgb[:] = [1.0, 0.5, 0.25]
        L.radius = 6.0
    return f


def views(gpu, ctx, f, size, chunk):
    """Two copies of the frame in one planned launch: pictures and totals."""
    targets = [gpu.Target(*size, depth=True, aux=False) for _ in range(2)]
    arr = (gpu.vrt_view * 2)()
    for v, t in zip(arr, targets):
        v.frame, v.target = f, t.struct()
    b = C.c_void_p()
    cfg = gpu.vrt_batch_config(8, 8, chunk, 0)
    gpu.call("vrt_batch_create", ctx.h, arr, 2, C.byref(cfg), C.byref(b))
    gpu.call("vrt_batch_launch", b)
    st = ctx.stats(reset=True)
    out = [t.download() for t in targets]
    gpu.call("vrt_batch_destroy", b)
    return out, st


@pytest.mark.parametrize("size", SMALL + LARGE, ids=lambda s: "%dx%d" % s)
def test_launch_shapes(gpu, orc, scene, size):
    dims, world, ctx = scene
    f = frame(gpu, dims, size)
    r = orc.render(world, dims, f, *size)
    totals = {}
    for cutoff in (False, True):  # off: the totals are the oracle's
        ctx.set_shadow_cutoff(cutoff)
        ctx.stats(reset=True)
        t = gpu.Target(*size, depth=True, aux=False)
        ctx.draw(t, frame=f)
        st = ctx.stats(reset=True)
        out = [t.download()]
        for chunk in (0, 3):
            o, s = views(gpu, ctx, f, size, chunk)
            out += o
            for k in ("rays", "dda_steps", "pixels"):
                assert s[k] == 2 * st[k], (cutoff, chunk, k, s[k], st[k])
        ctx.set_shadow_cutoff(True)
        assert st["pixels"] == size[0] * size[1] and st["rays"] == r["rays"]
        totals[cutoff] = st["dda_steps"]
        for i, o in enumerate(out):
            assert int(np.abs(o["rgb"].astype(np.int16) - r["rgb"].astype(np.int16)).max()) <= RGB_TOL, (cutoff, i)
            same = (o["depth"].view(np.uint32) == r["depth"].view(np.uint32)) | (np.isnan(o["depth"]) & np.isnan(r["depth"]))
            assert same.all(), (cutoff, i)
    assert totals[False] == r["dda_steps"] >= totals[True]


def test_walks_begun_again_count_once(gpu):
    """Where the wave's sum is counted (a plain draw beyond 16384 tiles, the
    hardware-scheduled views), a walk that run_walk gives up counts from then on
    in walk_generic; the persistent launch counts each lane's.  A scene that has
    such walks (its sun rays leave by the x-y edge), and others that reach the
    solid top at a whole y."""
    sc = gpu.make_scene("tiny", seed=1)
    size = (3840, 2160)
    f = sc.frame
    f.aspect_ratio = size[0] / size[1]
    ctx = gpu.Context(sc.dims)
    ctx.upload(sc.world)
    ctx.build_depth_field()
    out, lanes = views(gpu, ctx, f, size, 3)
    assert lanes["dda_steps"] > 3e8
    ctx.stats(reset=True)
    t = gpu.Target(*size, depth=True, aux=False)
    ctx.draw(t, frame=f)
    st = ctx.stats(reset=True)
    assert lanes["dda_steps"] == 2 * st["dda_steps"] and lanes["rays"] == 2 * st["rays"]
    assert np.array_equal(out[0]["rgb"], t.download()["rgb"])
    hw = views(gpu, ctx, f, size, 0)[1]
    assert hw["dda_steps"] == lanes["dda_steps"] and hw["rays"] == lanes["rays"]
    ctx.close()


def edge_scene(gpu, orc, dims, corner_words):
    """Jumps near the edge x = y = 0 and a camera whose rays all descend in x and
    y and leave there: many land with only x or only y below 0 and take their next
    step along the other axis.  The one solid voxel lies above the camera, so no
    ray takes the cutoff and the totals are the oracle's.  corner_words: some cells
    hold the guard corner's bits (a NaN jump, which ends a walk)."""
    rng = np.random.default_rng(5)
    cells = dims[0] * dims[1] * dims[2]
    world = np.full(cells, -1, np.int32)
    jump = rng.random(cells) < 0.6
    world[jump] = (-rng.uniform(0.5, 4.0, int(jump.sum())).astype(np.float32)).view(np.int32)
    if corner_words:
        world[rng.random(cells) < 0.05] = np.uint32(0xFFC00001).view(np.int32)
    world[cells - 1] = 0x334455
    f = gpu.frame_defaults(dims[0], 1024, 1024)
    f.cam_pos[:] = [6.3, 7.1, 0.4 * dims[2]]
    f.rotate_matrix[:] = gpu.camera_matrix(0.7, -0.5 * math.pi).tolist()
    f.focal = 3.0
    for vx in (-1.1, 1.1):  # beyond the widest picture below
        for vy in (-1.0, 1.0):
            d = orc.primary_dir(f, vx, vy)
            assert d[0] < -0.2 and d[1] < -0.2, d
    return world, f


@pytest.mark.parametrize("corner_words", [False, True], ids=["edge", "words"])
@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
def test_totals_of_walks_that_end_on_the_guard_corner(gpu, orc, dims, corner_words):
    """Totals of the wave's sum where run_walk's last word is the guard corner's
    and the shader's walk ends there too: the oracle's, and the persistent
    launch's lane by lane."""
    size = (1025, 1021)
    world, f = edge_scene(gpu, orc, dims, corner_words)
    f.aspect_ratio = size[0] / size[1]
    r = orc.render(world, dims, f, *size)
    assert r["rays"] == size[0] * size[1]  # every ray a miss
    ctx = gpu.Context(dims)
    ctx.upload(world)
    ctx.stats(reset=True)
    ctx.draw(gpu.Target(*size, depth=True, aux=False), frame=f)
    assert ctx.stats(reset=True)["dda_steps"] == r["dda_steps"]
    for chunk in (0, 3):
        assert views(gpu, ctx, f, size, chunk)[1]["dda_steps"] == 2 * r["dda_steps"], chunk
    ctx.close()


@pytest.fixture(scope="module")
def large(gpu):
    """A copy over 3.25 GiB that is at least 1400 long on x and z and 256 high."""
    dims = (1408, 256, 2400)
    p = gpu.world_params(dims, 3, caves=2000)
    ctx = gpu.Context(dims)
    ctx.generate(p)
    ctx.build_depth_field()
    yield dims, p, ctx, ctx.download()
    ctx.close()


@pytest.mark.parametrize("size", [(3, 8), (33, 8), (72, 56), (257, 131)], ids=lambda s: "%dx%d" % s)
@pytest.mark.parametrize("dist", [1399, 1400, 4000])
def test_far_views_in_four_wave_groups(gpu, orc, large, dist, size):
    """draw_form on either side of its render distance: a depth view and a step
    map, as a plain draw, hardware-scheduled and persistent views."""
    dims, p, ctx, words = large
    f = gpu.frame_defaults(dims[0], *size)
    x, z = dims[0] // 2, 200
    f.cam_pos[:] = [x + 0.3, gpu.surface(p, x, z) + 12.6, z + 0.4]
    f.rotate_matrix[:] = gpu.camera_matrix(0.05, 0.1).tolist()
    f.aspect_ratio = size[0] / size[1]
    f.render_dist = dist
    for depth_view in (1, 0):
        f.view_depth_field = depth_view
        t = gpu.Target(*size, depth=True, aux=True)
        ctx.stats(reset=True)
        ctx.draw(t, frame=f)
        st = ctx.stats(reset=True)
        g, r = t.download(), orc.render(words, dims, f, *size)
        for k in ("hit", "face", "steps", "shadow_eval", "shadow_occ"):
            assert np.array_equal(g[k], r[k]), (depth_view, k)
        assert int(np.abs(g["rgb"].astype(np.int16) - r["rgb"].astype(np.int16)).max()) <= RGB_TOL
        assert st["rays"] == r["rays"] and st["pixels"] == size[0] * size[1]
        if depth_view:  # no ray takes the cutoff
            assert st["dda_steps"] == r["dda_steps"]
            for chunk in (0, 3):
                out, s = views(gpu, ctx, f, size, chunk)
                assert all(np.array_equal(o["rgb"], g["rgb"]) for o in out), chunk
                assert s["dda_steps"] == 2 * st["dda_steps"] and s["pixels"] == 2 * st["pixels"], chunk
