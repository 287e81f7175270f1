"""The slot table and 9^3-voxel records that NanoVDB lookups read, bit for bit
against the oracle's tree walk at the borders of slots, blocks, regions and
constant tiles: the dense table, and the two-level one of a grid whose
clusters lie 4096 voxels apart on every axis."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT, TILE, UPPER, LOWER = 736, 32, 270400, 33856  # byte offsets / sizes of the 32.x records


def _grid(vrt, far):
    """Two root tiles along x (the second moved to 4096 on every axis if
    `far`), one constant upper-node tile and one constant lower-node tile."""
    rng = np.random.default_rng(5)
    dense = np.full((12, 10, 4104), 0.25, np.float32)
    for x in (slice(0, 20), slice(120, 140), slice(4090, 4104)):
        v = dense[:, :, x]
        m = rng.random(v.shape) < 0.3
        v[m] = rng.uniform(0.05, 1, m.sum())
    buf = vrt.gen_nanovdb_from_dense(dense, 0.25)
    assert buf[ROOT + 24:ROOT + 28].view(np.uint32)[0] == 2  # root tiles
    upper = ROOT + 64 + 2 * TILE
    lower = upper + 2 * UPPER
    n = 2 << 10  # region x in [256, 384): a constant tile
    at = upper + 8256 + 8 * n
    buf[at:at + 4].view(np.float32)[0] = 0.7
    n = 9 << 8 | 1 << 4  # slot (9, 1, 0) of region (0, 0, 0): a constant
    at = lower + 1088 + 8 * n
    buf[at:at + 4].view(np.float32)[0] = -0.5
    if far:
        key = ROOT + 64 + TILE
        buf[key:key + 8].view(np.uint64)[0] = 1 | 1 << 21 | 1 << 42
        buf[584:608].view(np.float64)[:] = (4105.0, 4107.0, 4109.0)
    return buf


@pytest.mark.parametrize("far", [False, True])
def test_lookup_tables(pkg, oracle, gpu_ctx, far):
    vrt = pkg.vrt
    buf = _grid(vrt, far)
    rng = np.random.default_rng(6)
    c = 4096.0 if far else 0.0
    boxes = [((-2, -2, -2), (22, 13, 15)), ((118, -2, -2), (142, 13, 15)),
             ((70, 6, -2), (82, 18, 10)), ((254, -3, 120), (260, 4, 131)),
             ((380, -3, -3), (387, 4, 4)), ((4088, -2, -2), (4106, 13, 15)),
             ((4094, c - 2, c - 2), (4106, c + 13, c + 15)), ((-9, -9, -9), (4200, 300, 300))]
    pts = np.concatenate([rng.uniform(lo, hi, (4000, 3)) for lo, hi in boxes]
                         + [rng.integers(-2, 30, (500, 3)), [[np.nan, 1, 1], [1e30, 0, 0],
                                                            [np.inf, 2, 2], [-3e9, 4, 4]]])
    pts = pts.astype(np.float32)
    tf = pkg.workloads.albedo_tf(0.8, 64)
    for filt in ("linear", "nearest"):
        dv = vrt.DeviceVolume.from_nanovdb(gpu_ctx, buf, tf, (0, 1), 1.0, None, filter=filt)
        g = vrt.sample_field(gpu_ctx, dv, pts)
        o = oracle.nvdb_sample(buf, pts[:-4], 1 if filt == "linear" else 0)
        np.testing.assert_array_equal(g[:-4], o)
        # no voxel there: the background, NaN where an interpolation weight is
        assert g[-3] == 0.25 and g[-1] == 0.25
        if filt == "linear":
            assert np.isnan(g[-4]) and np.isnan(g[-2])
        assert len(np.unique(o)) > 1000 and (o == 0.7).any() and (o == -0.5).any()


def _check(pkg, oracle, ctx, grid, buf, pts):
    vrt = pkg.vrt
    pts = np.concatenate(pts).astype(np.float32)
    tf = pkg.workloads.albedo_tf(0.8, 64)
    for filt in ("linear", "nearest"):
        dv = vrt.DeviceVolume.from_nanovdb(ctx, grid, tf, (0, 1), 1.0, None, filter=filt)
        o = oracle.nvdb_sample(buf, pts, 1 if filt == "linear" else 0)
        np.testing.assert_array_equal(vrt.sample_field(ctx, dv, pts), o)
    return o


def test_wide_tile_borders(pkg, oracle, gpu_ctx):
    """A 4096^3 constant root tile beside an upper node with 512 constant
    tiles of values of their own: memory goes with the tree's nodes, not with
    the surface of its tiles (1.6 M slots lie along the root tile's)."""
    vrt = pkg.vrt
    rng = np.random.default_rng(8)
    dense = np.zeros((9, 9, 4100), np.float32)
    dense[:, :, :9] = rng.uniform(0.1, 1, (9, 9, 9))
    dense[0, 0, 4099] = 1.0
    buf = vrt.gen_nanovdb_from_dense(dense, 0.0)
    assert buf[ROOT + 24:ROOT + 28].view(np.uint32)[0] == 2  # root tiles
    tile = ROOT + 64 + TILE  # x in [4096, 8192)
    buf[tile + 8:tile + 16].view(np.int64)[0] = 0
    buf[tile + 20:tile + 24].view(np.float32)[0] = 0.625
    upper = ROOT + 64 + 2 * TILE
    for x in range(4, 12):
        for y in range(4, 12):
            for z in range(4, 12):
                at = upper + 8256 + 8 * (x << 10 | y << 5 | z)
                buf[at:at + 4].view(np.float32)[0] = rng.uniform(0.1, 1)
    buf[584:608].view(np.float64)[:] = (8192.0, 4096.0, 4096.0)
    grid = vrt.DeviceNanoVDB(gpu_ctx, buf)
    assert grid.info.device_bytes < 16 << 20
    pts = [rng.uniform(-2, 20, (4000, 3)), rng.uniform(500, 1600, (20000, 3)),
           rng.uniform((-9, -9, -9), (8200, 4100, 4100), (20000, 3))]
    # on and around the borders of the tiles: faces, edges and corners
    edges = 128 * rng.integers(3, 14, (20000, 3)) + rng.choice([-1, 0, 0.25, 7.5, 64.5], (20000, 3))
    pts += [edges, edges + rng.uniform(-1.5, 1.5, edges.shape)]
    root = np.array((4096.0, 0.0, 0.0)) + 4096 * rng.integers(0, 2, (20000, 3))
    pts.append(np.where(rng.random(root.shape) < 0.6, root + rng.uniform(-1.5, 1.5, root.shape),
                        rng.uniform(0, 8192, root.shape)))
    o = _check(pkg, oracle, gpu_ctx, grid, buf, pts)
    assert (o == np.float32(0.625)).sum() > 1000 and len(np.unique(o)) > 500


def test_leaves_apart(pkg, oracle, gpu_ctx):
    """4096 leaves that touch no other would take 8 records each: lookups walk
    the tree, in the dense table and behind the region table."""
    vrt = pkg.vrt
    rng = np.random.default_rng(9)
    dense = np.zeros((256, 256, 256), np.float32)
    v = dense.reshape(16, 16, 16, 16, 16, 16)[:, :8, :, :8, :, :8]  # every other slot
    v[...] = np.where(rng.random(v.shape) < 0.5, rng.uniform(0.1, 1, v.shape), 0)
    far = np.zeros((256, 256, 4097), np.float32)
    far[:, :, :256] = dense
    far[0, 0, 4096] = 0.5
    for vox, n in ((dense, 256), (far, 256)):
        buf = vrt.gen_nanovdb_from_dense(vox, 0.0)
        if vox is far:  # (the second root tile far away on every axis)
            buf[ROOT + 64 + TILE:ROOT + 72 + TILE].view(np.uint64)[0] = 1 | 1 << 21 | 1 << 42
            buf[584:608].view(np.float64)[:] = (4098.0, 4098.0, 4098.0)
        grid = vrt.DeviceNanoVDB(gpu_ctx, buf)
        assert grid.info.leaves >= 4096
        assert grid.info.device_bytes < 2 * buf.nbytes
        edges = 8 * rng.integers(-1, 34, (20000, 3)) + rng.choice([-1, 0, 0.25], (20000, 3))
        pts = [rng.uniform(-9, n + 9, (40000, 3)), edges,
               edges + rng.uniform(-1.5, 1.5, edges.shape), rng.uniform(4090, 4100, (500, 3))]
        o = _check(pkg, oracle, gpu_ctx, grid, buf, pts)
        assert len(np.unique(o)) > 2000
