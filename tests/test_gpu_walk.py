"""The written-out walk (vrt_device.h: cast_ray, run_walk) where its arithmetic
differs in form from the shader's: whole coordinates after a jump, ties, walks
that leave the grid by a low face or by the x-y edge, starts outside its range,
directions so long that a jump ends beyond 2^31, components near 0.
Against the oracle's castRay, bit for bit, for 32-bit byte offsets and 32-bit
indices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(24, 20, 40), (4096, 600, 2)]  # byte offsets; 4 X Y >= 2^23: word indices


def compare(gpu, orc, world, dims, start, d, dist, budget=256):
    start, d = np.asarray(start, np.float32), np.asarray(d, np.float32)
    dist = np.asarray(dist, np.int32)
    ctx = gpu.Context(dims)
    ctx.upload(world)
    r = orc.cast_rays(world, dims, start, d, dist, budget)
    for steps in (True, False):
        g = ctx.cast_rays(start, d, dist, budget, steps=steps)
        for k in ("hit", "face", "steps") if steps else ("hit", "face"):
            bad = np.nonzero(g[k] != r[k])[0]
            assert bad.size == 0, "%s differs for %d rays, first start %s dir %s: %s, oracle %s" % (
                k, bad.size, start[bad[0]].tolist(), d[bad[0]].tolist(), g[k][bad[0]], r[k][bad[0]])
        # bitwise, any NaN equal to any NaN
        same = (g["hit_pos"].view(np.uint32) == r["hit_pos"].view(np.uint32)) | (np.isnan(g["hit_pos"]) & np.isnan(r["hit_pos"]))
        bad = np.nonzero(~same.all(1))[0]
        assert bad.size == 0, "hit_pos differs for %d rays, first start %s dir %s: %s, oracle %s" % (
            bad.size, start[bad[0]].tolist(), d[bad[0]].tolist(), g["hit_pos"][bad[0]], r["hit_pos"][bad[0]])
    ctx.close()
    return r


@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
@pytest.mark.parametrize("seed", [1, 2, 3])
def test_walks_on_dyadic_numbers(gpu, orc, dims, seed):
    """Starts, directions and jumps that are small multiples of powers of two:
    every product and sum is exact, so coordinates after a jump are often whole
    and intersects often equal."""
    rng = np.random.default_rng(seed)
    X, Y, Z = dims
    cells = X * Y * Z
    world = np.full(cells, -1, np.int32)
    jump = rng.random(cells) < 0.5
    world[jump] = (-0.5 * rng.integers(1, 17, int(jump.sum())).astype(np.float32)).view(np.int32)
    solid = rng.random(cells) < 0.04
    world[solid] = rng.integers(0, 1 << 24, int(solid.sum()))
    n = 40000
    start = np.stack([rng.integers(0, 4 * min(s, 48), n) / 4.0 for s in dims], 1)
    start += rng.choice([0.0, 0.0, 0.5, 2.0 ** -20, 2.0 ** -21], (n, 1))
    far = rng.random(n) < 0.3  # near the high faces
    start[far] = np.array(dims) - start[far]
    d = rng.choice([-1.0, -0.5, -0.25, 0.25, 0.5, 1.0], (n, 3))
    some = rng.random(n) < 0.1
    d[some, rng.integers(0, 3)] = 0.0
    r = compare(gpu, orc, world, dims, start, d, rng.integers(1, 200, n))
    assert int((r["hit"] >= 0).sum()) > 1000  # 5-6% of the rays on the flat grid


def test_leaving_by_the_edge_with_equal_intersects(gpu, orc):
    """A jump that leaves x and y in (-1, 0), both heading down, with equal
    (negative) intersects: the shader steps z and stays in the cell column
    x = y = 0 until a solid voxel, a jump or the grid's end."""
    dims = (12, 12, 40)
    X, Y, _ = dims
    starts, dirs, worlds = [], [], []
    for dz in (0.3, -0.3):
        for zs in (1, 2, 5):  # z steps from the jump's end to the solid voxel
            z0 = 5.5 if dz > 0 else 30.5
            w = np.full(dims[0] * dims[1] * dims[2], -1, np.int32)
            first = 6 if dz > 0 else 29  # x and y tie at the start too: z is stepped
            w[2 + X * 2 + X * Y * first] = np.float32(-(6.0 - 0.5 / 0.3)).view(np.int32)
            end = int(z0 + dz * 6.0)
            w[X * Y * (end + (zs if dz > 0 else -zs))] = 0x112233
            starts.append([2.5, 2.5, z0])
            dirs.append([-0.5, -0.5, dz])
            worlds.append(w)
    hits = 0
    for s, d, w in zip(starts, dirs, worlds):
        n = 70  # more than one wave, the other lanes on other walks
        start = np.repeat(np.array([s]), n, 0)
        start[1::2, 0] += np.linspace(0.1, 3.0, n)[1::2]
        r = compare(gpu, orc, w, dims, start, np.repeat(np.array([d]), n, 0), np.full(n, 200))
        hits += int((r["hit"][::2] >= 0).sum())
    assert hits == 6 * 35, hits  # every such ray reaches its voxel


def jumps_and_solids(rng, dims):
    cells = dims[0] * dims[1] * dims[2]
    world = np.full(cells, -1, np.int32)
    jump = rng.random(cells) < 0.5
    world[jump] = (-0.5 * rng.integers(1, 17, int(jump.sum())).astype(np.float32)).view(np.int32)
    solid = rng.random(cells) < 0.04
    world[solid] = rng.integers(0, 1 << 24, int(solid.sum()))
    return world


@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
@pytest.mark.parametrize("axis", [0, 1, 2, None], ids=["x", "y", "z", "all"])
def test_long_directions(gpu, orc, dims, axis):
    """One component of 2^20 to 2^60, or each of 2^-19 to 2^60: most jumps end far
    outside the grid, many beyond 2^31, where the cell saturates; the walk has to
    leave the grid there, one iteration later.  (run_walk takes none of the first,
    and of the others those up to 2^6.)"""
    rng = np.random.default_rng(40 if axis is None else 41 + axis)
    world = jumps_and_solids(rng, dims)
    n = 40000
    start = np.stack([rng.uniform(0.01, min(s, 48), n) for s in dims], 1)
    d = rng.choice([-1.0, 1.0], (n, 3)) * 2.0 ** rng.uniform(-8, 2, (n, 3))
    if axis is None:
        d = rng.choice([-1.0, 1.0], (n, 3)) * 2.0 ** rng.uniform(-19, 60, (n, 3))
    else:
        d[:, axis] = rng.choice([-1.0, 1.0], n) * 2.0 ** rng.uniform(20, 60, n)
    compare(gpu, orc, world, dims, start, d, rng.integers(1, 200, n))


@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
def test_components_near_zero(gpu, orc, dims):
    """Components on both sides of 2^-60 and 2^-19, and around the -1e-6 whose
    step size is infinite; starts near the low faces."""
    rng = np.random.default_rng(47)
    world = jumps_and_solids(rng, dims)
    n = 40000
    start = np.stack([rng.uniform(2.0 ** -20, min(s, 48), n) for s in dims], 1)
    low = rng.random((n, 3)) < 0.1
    start[low] = 2.0 ** rng.uniform(-20, 0, int(low.sum()))
    d = rng.normal(size=(n, 3))
    small = rng.random((n, 3)) < 0.3
    d[small] = rng.choice([-1.0, 1.0], int(small.sum())) * 2.0 ** rng.uniform(-62, -12, int(small.sum()))
    step = rng.random((n, 3)) < 0.05
    d[step] = np.float32(-1e-6) * (1 + rng.integers(-4, 5, int(step.sum())) * 2.0 ** -23)
    r = compare(gpu, orc, world, dims, start, d, rng.integers(1, 200, n))
    assert int((r["hit"] >= 0).sum()) > 1000


@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
def test_longest_jumps_that_run_walk_takes(gpu, orc, dims):
    """Components up to 2^6, jumps and budgets up to 2^24: positions up to 2^30,
    short of where a cell saturates."""
    rng = np.random.default_rng(46)
    cells = dims[0] * dims[1] * dims[2]
    world = np.full(cells, -1, np.int32)
    jump = rng.random(cells) < 0.3
    world[jump] = (-(2.0 ** rng.uniform(0, 24, int(jump.sum()))).astype(np.float32)).view(np.int32)
    solid = rng.random(cells) < 0.04
    world[solid] = rng.integers(0, 1 << 24, int(solid.sum()))
    n = 40000
    start = np.stack([rng.uniform(0.01, min(s, 48), n) for s in dims], 1)
    d = rng.choice([-1.0, 1.0], (n, 3)) * np.minimum(2.0 ** rng.uniform(-19, 8, (n, 3)), 2.0 ** 6)
    compare(gpu, orc, world, dims, start, d, np.full(n, 1 << 24), 1 << 24)


def test_step_count_of_a_jump_beyond_two_to_the_31(gpu, orc):
    """Two iterations: the step into the jump, then the one that leaves the grid
    from beyond y = 2^31."""
    dims = (24, 20, 40)
    world = np.full(dims[0] * dims[1] * dims[2], -1, np.int32)
    world[5 + dims[0] * (6 + dims[1] * 5)] = np.float32(-2.0).view(np.int32)
    r = compare(gpu, orc, world, dims, [[5.5, 5.5, 5.5]], [[0.3, 2.0 ** 32, 0.3]], [200], 200)
    assert r["steps"].tolist() == [2]


@pytest.mark.parametrize("dims", GRIDS, ids=["byte_offset32", "index32"])
@pytest.mark.parametrize("axis", [0, 1, 2], ids="xyz")
def test_primary_rays_with_a_component_near_zero(gpu, orc, dims, axis):
    """Frames whose rays all have one small component, down to below 2^-60, by a
    scaled rotation; or one near the -1e-6 whose step size is infinite."""
    rng = np.random.default_rng(48 + axis)
    world = jumps_and_solids(rng, dims)
    ctx = gpu.Context(dims)
    ctx.upload(world)
    size = (72, 56)
    t = gpu.Target(*size, depth=True, aux=True)
    hits = 0
    for scale in [2.0 ** -k for k in (10, 19, 21, 35, 50, 58, 62)] + [-1e-6]:
        f = gpu.frame_defaults(dims[0], *size)
        f.cam_pos[:] = [0.4 * dims[0], 0.5 * dims[1], 0.3 * dims[2]]
        m = np.asarray(gpu.camera_matrix(0.3, 0.7), np.float32).reshape(4, 4)  # columns
        m[:3, axis] *= np.float32(scale)
        if scale < 0:  # -1e-6 times the depth component of the pixel
            m[:3, axis] = 0.0
            m[2, axis] = np.float32(scale)
        f.rotate_matrix[:] = m.ravel().tolist()
        f.aspect_ratio = size[0] / size[1]
        for depth_view in (0, 1):
            f.view_depth_field = depth_view
            ctx.draw(t, frame=f)
            g, r = t.download(), orc.render(world, dims, f, *size)
            for k in ("hit", "face", "steps", "shadow_eval", "shadow_occ"):
                bad = np.argwhere(g[k] != r[k])
                assert bad.size == 0, (scale, depth_view, k, len(bad), bad[0].tolist())
            same = (g["depth"].view(np.uint32) == r["depth"].view(np.uint32)) | (np.isnan(g["depth"]) & np.isnan(r["depth"]))
            assert same.all(), (scale, depth_view)
        hits += int((r["hit"] >= 0).sum())
    assert hits > 500
    ctx.close()
