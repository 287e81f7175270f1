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
