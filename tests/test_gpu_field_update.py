"""Field preparation kernels against numpy at the edges of their tiles:
brick records (runs of 8 bricks along x, 9^3 records), macrocell value
ranges (rows packed into waves) and majorants (16-entry blocks of the TF)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def records(vox):
    """Brick records of (nz, ny, nx) voxels, clamp addressing."""
    idx = [np.minimum(np.arange(-(-n // 8))[:, None] * 8 + np.arange(9), n - 1) for n in vox.shape]
    b = vox[idx[0]][:, :, idx[1]][:, :, :, :, idx[2]]  # bz 9 by 9 bx 9
    b = b.transpose(0, 2, 4, 1, 3, 5).reshape(-1, 729)
    return np.pad(b, ((0, 0), (0, 7))).ravel()


def footprints(n, G):
    """The voxel range [a, e] a trilinear sample in each of G cells can read."""
    return [(max(0, int(np.floor(m * n / G - 0.5))),
             min(n - 1, int(np.floor((m + 1) * n / G - 0.5)) + 1)) for m in range(G)]


@pytest.mark.parametrize("dims,grid,tf_size", [
    ((1, 1, 1), (1, 1, 1), 1), ((8, 8, 8), (1, 1, 1), 16), ((9, 17, 65), (1, 2, 5), 17),
    ((64, 9, 8), (4, 1, 1), 255), ((65, 63, 20), (5, 4, 2), 4096), ((130, 7, 5), (1, 1, 1), 5000),
    ((5, 3, 4), (7, 8, 9), 33), ((257, 33, 31), (16, 2, 3), 256)])
def test_bricks_ranges_majorants(pkg, gpu_ctx, dims, grid, tf_size):
    vrt = pkg.vrt
    ctx = gpu_ctx
    rng = np.random.default_rng(dims[0])
    vox = rng.random(dims[::-1], np.float32)
    tf = rng.random((tf_size, 4), np.float32)
    tf[rng.random(tf_size) < 0.5, 3] = 0.0
    dv = vrt.DeviceVolume(ctx, vox, (0, 0, 0), (1, 1, 1), tf, (0.2, 0.9), 1.0, grid)
    exp = records(vox)
    np.testing.assert_array_equal(dv.bricks.download(np.float32, exp.shape), exp)

    got = dv.ranges.download(np.float32, (int(np.prod(grid)), 2))
    maj = dv.majorants.download(np.float32, (int(np.prod(grid)),))
    step = dv.majorant_step.download(np.float32, (1,))[0]
    assert step * np.float32(255) >= tf[:, 3].max()
    fx, fy, fz = (footprints(n, G) for n, G in zip(dims, grid))
    f32, n = np.float32, tf_size
    for c in range(len(got)):
        x, y, z = c % grid[0], (c // grid[0]) % grid[1], c // (grid[0] * grid[1])
        box = vox[fz[z][0]:fz[z][1] + 1, fy[y][0]:fy[y][1] + 1, fx[x][0]:fx[x][1] + 1]
        assert got[c, 0] == box.min() and got[c, 1] == box.max(), c
        taps = []
        for v, up in ((box.min(), 0), (box.max(), 1)):
            u = (v - f32(0.2)) / (f32(0.9) - f32(0.2))
            t = min(max(u * f32(n) - f32(0.5), f32(-1)), f32(n))
            taps.append(min(max(int(np.floor(t)) + up, 0), n - 1))
        m = max(f32(0), tf[taps[0]:taps[1] + 1, 3].max())
        q = 0
        if m > 0:
            q = int(min(f32(255), np.ceil(m / step)))
            while q < 255 and f32(q) * step < m:
                q += 1
        assert maj[c] == f32(q) * step, c


@pytest.mark.parametrize("cell,grid", [(c, (3, 2, 2)) for c in (1, 2, 3, 4, 5, 7, 8, 11, 16, 21,
                                                                33, 66)]
                         + [(c, (17, 16, 16)) for c in (1, 4, 8, 14, 15)] + [(8, (17, 16, 15))])
def test_value_ranges_of_cell_sizes(pkg, gpu_ctx, cell, grid):
    """Footprints from 2 to 68 voxels a side, few cells and more than 4096:
    one wave or four per cell, lanes with one row, some, and several batches."""
    vrt = pkg.vrt
    dims = tuple(max(1, g * cell - a) for a, g in enumerate(grid))
    vox = np.random.default_rng(cell).normal(size=dims[::-1]).astype(np.float32)
    dv = vrt.DeviceVolume(gpu_ctx, vox, (0, 0, 0), (1, 1, 1), np.ones((2, 4), np.float32), (0, 1),
                          1.0, grid)
    got = dv.ranges.download(np.float32, grid[::-1] + (2,))
    lo = hi = vox
    for axis in range(3):
        f = footprints(dims[2 - axis], grid[2 - axis])
        lo = np.stack([lo.take(range(a, e + 1), axis).min(axis) for a, e in f], axis)
        hi = np.stack([hi.take(range(a, e + 1), axis).max(axis) for a, e in f], axis)
    np.testing.assert_array_equal(got[..., 0], lo)
    np.testing.assert_array_equal(got[..., 1], hi)


@pytest.mark.parametrize("dims", [(1, 1, 1), (8, 9, 7), (16, 17, 300), (9, 1000, 200), (17, 520, 440),
                                  (25, 400, 330), (112, 110, 112), (120, 128, 129), (100, 3, 4096)])
def test_brick_records_of_sizes(pkg, gpu_ctx, dims):
    """Brick records one per workgroup and in runs: either side of 3,072
    bricks, and one to four bricks along x."""
    vox = np.random.default_rng(dims[0]).random(dims[::-1], np.float32)
    dv = pkg.vrt.DeviceVolume(gpu_ctx, vox, (0, 0, 0), (1, 1, 1), np.ones((2, 4), np.float32),
                              (0, 1), 1.0)
    exp = records(vox)
    np.testing.assert_array_equal(dv.bricks.download(np.float32, exp.shape), exp)
