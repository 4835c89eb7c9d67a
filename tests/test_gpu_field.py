"""The bit-parallel depth field (vrt_field.h) against the oracle's
fixDepthField, word for word: sizes around the tile (32 x 8 x 16 voxels) and
the bitmap's words, densities from one solid voxel to nearly full, and empty
voxels that already hold other words.  The padded copy that the build writes
is read back through rays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_world(rng, dims, density):
    n = dims[0] * dims[1] * dims[2]
    w = np.full(n, -1, np.int32)
    # empty voxels holding some jump already: nearer than 2 cells they keep it
    old = rng.random(n) < 0.3
    w[old] = (-np.sqrt(rng.integers(4, 37, int(old.sum())).astype(np.float32))).view(np.int32)
    solid = rng.random(n) < density
    solid[rng.integers(0, n)] = True
    w[solid] = rng.integers(0, 1 << 24, int(solid.sum()))
    return w


def check_rays(gpu, orc, ctx, words, dims, rng, n=4000):
    start = np.stack([rng.uniform(-1.5, d + 1.5, n) for d in dims], 1).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    dist = rng.integers(1, 200, n).astype(np.int32)
    g = ctx.cast_rays(start, d, dist, 256)
    r = orc.cast_rays(words, dims, start, d, dist, 256)
    for k in ("hit", "face", "steps"):
        assert np.array_equal(g[k], r[k]), "%s differs for %d rays" % (k, int((g[k] != r[k]).sum()))


DIMS = [(1, 1, 1), (31, 7, 15), (32, 8, 16), (33, 9, 17), (34, 8, 16), (63, 16, 33), (64, 15, 32), (65, 17, 31),
        (66, 3, 50), (127, 25, 2), (130, 40, 47), (16, 30, 64), (5, 64, 5)]


@pytest.mark.parametrize("dims", DIMS, ids=["%dx%dx%d" % d for d in DIMS])
@pytest.mark.parametrize("density", [0.0, 0.002, 0.05, 0.97])
def test_build_equals_oracle(gpu, orc, dims, density):
    rng = np.random.default_rng(dims[0] * 7919 + dims[1] * 31 + dims[2] + int(density * 1000))
    world = random_world(rng, dims, density)
    ctx = gpu.Context(dims)
    ctx.upload(world)
    ctx.build_depth_field()
    got, ref = ctx.download(), orc.depth_field(world, dims)
    assert np.array_equal(got, ref), "%d voxels differ" % int((got != ref).sum())
    check_rays(gpu, orc, ctx, ref, dims, rng)
    ctx.close()


def test_build_around_one_voxel_at_every_place_in_a_tile(gpu, orc):
    """One solid voxel, at places that cover every x in a bitmap word and every
    (y, z) of a tile: all distance classes, across every kind of tile border."""
    dims = (96, 24, 48)
    ctx = gpu.Context(dims)
    for k in range(32):
        x, y, z = 32 + k, 8 + k % 8, 16 + (k * 5) % 16
        world = np.full(dims[0] * dims[1] * dims[2], -1, np.int32)
        world[x + dims[0] * (y + dims[1] * z)] = 0x203040
        ctx.upload(world)
        ctx.build_depth_field()
        got, ref = ctx.download(), orc.depth_field(world, dims)
        assert np.array_equal(got, ref), "voxel (%d, %d, %d): %d differ" % (x, y, z, int((got != ref).sum()))
    ctx.close()


def build(gpu, orc, dims, density, seed):
    rng = np.random.default_rng(seed)
    world = random_world(rng, dims, density)
    ctx = gpu.Context(dims)
    ctx.upload(world)
    ctx.build_depth_field()
    return rng, ctx, orc.depth_field(world, dims)


@pytest.mark.parametrize("radius", [-3, -2, -1, 0, 1, 2, 5, 8, 13, 14, 40])
@pytest.mark.parametrize("density", [0.01, 0.6])
def test_remove_sphere_equals_oracle(gpu, orc, radius, density):
    """Carve, repair and render copy in one launch: boxes of one and several
    tiles (32 x 8 x 8), clipped at corners and faces, overlapping, with centres
    in and outside the grid."""
    dims = (75, 41, 58)
    rng, ctx, ref = build(gpu, orc, dims, density, 100 + radius)
    centres = [(0, 0, 0), (dims[0] - 1, dims[1] - 1, dims[2] - 1), (37, 20, 29), (38, 21, 30), (-2, 20, 70),
               (31, 8, 8)] + [tuple(int(rng.integers(0, d)) for d in dims) for _ in range(3)]
    for c in centres:
        orc.remove_sphere(ref, dims, c, radius)
        ctx.remove_sphere(*c, radius)
    got = ctx.download()
    assert np.array_equal(got, ref), "%d voxels differ" % int((got != ref).sum())
    check_rays(gpu, orc, ctx, ref, dims, rng)
    ctx.close()


@pytest.mark.parametrize("lo,hi", [((0, 0, 0), (75, 41, 58)), ((5, 3, 9), (6, 4, 10)), ((10, 7, 1), (43, 16, 9)),
                                   ((-9, 30, 40), (200, 90, 99)), ((33, 1, 1), (33, 9, 9))])
def test_fix_box_equals_oracle(gpu, orc, lo, hi):
    dims = (75, 41, 58)
    rng = np.random.default_rng(sum(lo) + sum(hi))
    world = random_world(rng, dims, 0.03)
    ctx = gpu.Context(dims)
    ctx.upload(world)
    ctx.fix_depth_field_box(lo, hi)
    box = tuple(slice(max(0, lo[k]), max(0, min(dims[k], hi[k]))) for k in (2, 1, 0))
    ref = world.copy()
    ref.reshape(dims[::-1])[box] = orc.depth_field(world, dims).reshape(dims[::-1])[box]
    got = ctx.download()
    assert np.array_equal(got, ref), "%d voxels differ" % int((got != ref).sum())
    check_rays(gpu, orc, ctx, ref, dims, rng)
    ctx.close()


@pytest.mark.parametrize("lo,size", [((3, 2, 1), (1, 1, 1)), ((0, 0, 0), (10, 10, 10)), ((255, 30, 190), (1, 70, 60)),
                                     ((0, 0, 0), (256, 64, 16)), ((0, 0, 0), (256, 64, 32)), ((1, 0, 3), (255, 90, 77)),
                                     ((0, 0, 0), (256, 129, 250))])
def test_region_upload_in_pieces(gpu, orc, lo, size):
    """Partial uploads of less than, exactly and more than the staging's pieces
    (2^18 words), pieces that end inside a row; the solid top follows."""
    dims = (256, 130, 251)
    rng = np.random.default_rng(size[0] + size[1])
    ctx = gpu.Context(dims)
    host = random_world(rng, dims, 0.01)
    hi = tuple(lo[k] + size[k] - (k == 0) for k in range(3))  # inside the grid, or the corners would be swapped
    ctx.upload_region(host, lo, hi)
    ref = np.full_like(host, -1)
    box = tuple(slice(lo[k], lo[k] + size[k]) for k in (2, 1, 0))
    ref.reshape(dims[::-1])[box] = host.reshape(dims[::-1])[box]
    got = ctx.download()
    assert np.array_equal(got, ref), "%d voxels differ" % int((got != ref).sum())
    check_rays(gpu, orc, ctx, ref, dims, rng)
    # rays that rise take the cutoff at the solid top when no steps are asked for
    n = 4000
    start = np.stack([rng.uniform(0, d, n) for d in dims], 1).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d[:, 1] = np.abs(d[:, 1])
    dist = np.full(n, 300, np.int32)
    g, r = ctx.cast_rays(start, d, dist, 384, steps=False), orc.cast_rays(ref, dims, start, d, dist, 384)
    assert np.array_equal(g["hit"], r["hit"])
    ctx.close()


@pytest.mark.parametrize("dims", DIMS, ids=["%dx%dx%d" % d for d in DIMS])
def test_device_upload_at_odd_sizes(gpu, orc, dims):
    """vrt_upload_device: grid, render copy and solid top in one pass, rows of
    every length modulo four and grids of few rows."""
    rng = np.random.default_rng(sum(dims))
    world = random_world(rng, dims, 0.02)
    ctx = gpu.Context(dims)
    buf = gpu.DeviceBuffer(world.nbytes)
    buf.upload(world)
    gpu.call("vrt_upload_device", ctx.h, buf.addr)
    assert np.array_equal(ctx.download(), world)
    check_rays(gpu, orc, ctx, world, dims, rng)
    n = 2000
    start = np.stack([rng.uniform(0, d, n) for d in dims], 1).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    d[:, 1] = np.abs(d[:, 1])
    dist = np.full(n, 300, np.int32)
    g, r = ctx.cast_rays(start, d, dist, 384, steps=False), orc.cast_rays(world, dims, start, d, dist, 384)
    assert np.array_equal(g["hit"], r["hit"])
    ctx.close()
