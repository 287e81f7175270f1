"""Traversal against brute force for trees whose deepest lists are cut by
count, not by the sweep: a leaf's triangle count has one byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tail", [200, 255, 256, 700])
def test_long_lists_below_level_60(pkg, oracle, gpu_ctx, tail):
    vrt = pkg.vrt
    rng = np.random.default_rng(tail)
    # centroids at 2^-i: a level of the sweep peels off the farthest few
    x = np.concatenate([2.0 ** -np.arange(100), 2.0 ** -100 * (1 + rng.random(tail))])
    # triangles across the x axis whose box centres differ in x alone
    h = rng.uniform(0.02, 0.05, (len(x), 2))
    tri = np.zeros((len(x), 3, 3))
    tri[:, :, 0] = x[:, None]
    tri[:, :, 1] = h[:, :1] * [-1, 1, 0]
    tri[:, :, 2] = h[:, 1:] * [-1, -1, 1]
    v = tri.astype(np.float32).reshape(-1, 3)
    mesh = vrt.DeviceMesh(gpu_ctx, v, None, "sah")
    scene = vrt.make_scene([], [], [(mesh, (0.7, 0.7, 0.7))])
    r = np.zeros((6000, 8), np.float32)
    r[:, 7] = 1e30
    r[:2000, 0:3] = rng.uniform(-1, 2, (2000, 3))
    at = v.reshape(-1, 3, 3).mean(1)[rng.integers(0, len(x), 2000)]
    r[:2000, 3:6] = at - r[:2000, 0:3]
    # (from below, the tail's triangles are hit at one distance: the lowest wins)
    r[2000:, 0:3] = np.where(np.arange(4000)[:, None] % 2, (2.0, 0.0, 0.0), (-1.0, 0.0, 0.0))
    r[2000:, 3:6] = np.where(np.arange(4000)[:, None] % 2, (-1.0, 0.0, 0.0), (1.0, 0.0, 0.0))
    r[2000:, 4:6] += rng.normal(0, 0.01, (4000, 2))
    r[:, 3:6] /= np.linalg.norm(r[:, 3:6], axis=1, keepdims=True)
    om = oracle.OracleMesh(v, None)
    t, p = vrt.intersect_surfaces(gpu_ctx, scene, r, False)
    to, po = oracle.mesh_intersect(om, r, any_hit=False, brute=True)
    # the tail's triangles lie in one plane to within 2^-100, so their computed
    # distances differ by rounding alone: t = dot(e2, s2) / dot(s1, e1), two sums
    # of three products of twice rounded factors, some 8 roundings of 2^-24
    # each, 1e-6 in all; the traversal culls boxes beyond the closest hit with a
    # slack of 2e-7 and need not meet the one whose distance rounds lowest
    np.testing.assert_array_equal(p >= 0, po >= 0)
    np.testing.assert_allclose(t[po >= 0], to[po >= 0], rtol=1e-6)
    apart = (po >= 0) & (po < 50)  # planes that distances tell apart
    near = t != to
    assert np.mean(p[apart] == po[apart]) >= 0.999 and near.mean() <= 1e-3
    ta, pa = vrt.intersect_surfaces(gpu_ctx, scene, r, True)
    np.testing.assert_array_equal(pa >= 0, po >= 0)
    assert (po >= 0).mean() > 0.05


@pytest.mark.parametrize("count", [1, 2, 3, 4])
def test_any_hit_returns_the_first_of_a_leaf(pkg, gpu_ctx, count):
    """Up to 4 triangles are one leaf, held in the order given: an any-hit
    call returns the first that the ray meets, whatever lies nearer."""
    vrt = pkg.vrt
    tri = np.zeros((count, 3, 3), np.float32)
    for i in range(count):  # planes z = -i; the first ones also narrower in x
        tri[i] = [(-2 - i, -2, -i), (2 + i, -2, -i), (0, 4 + 2 * i, -i)]
    mesh = vrt.DeviceMesh(gpu_ctx, tri.reshape(-1, 3), None, "sah")  # (outlives the scene)
    scene = vrt.make_scene([], [], [(mesh, (0.7, 0.7, 0.7))])
    rng = np.random.default_rng(count)
    r = np.zeros((4000, 8), np.float32)
    r[:, :3] = rng.uniform(-5, 5, (4000, 3))
    r[:, 2] = np.where(np.arange(4000) % 2, 3.0, -7.0)
    r[:, 5] = np.where(np.arange(4000) % 2, -1.0, 1.0)
    r[:, 7] = 1e30
    hit = np.stack([(r[:, 1] > -2) & (r[:, 1] < (4 + 2 * i) - (6 + 2 * i) * np.abs(r[:, 0]) / (2 + i))
                    for i in range(count)])
    # (edges: no ray within 1e-3 of one)
    edge = np.stack([np.minimum(np.abs(r[:, 1] + 2), np.abs(
        (4 + 2 * i) - (6 + 2 * i) * np.abs(r[:, 0]) / (2 + i) - r[:, 1])) for i in range(count)])
    keep = edge.min(0) > 1e-3
    first = np.where(hit.any(0), hit.argmax(0), -1)
    t, p = vrt.intersect_surfaces(gpu_ctx, scene, r, True)
    np.testing.assert_array_equal(p[keep], first[keep])
    got = keep & (first >= 0)
    np.testing.assert_allclose(t[got], np.abs(r[got, 2] + first[got]), rtol=1e-5)
    assert got.sum() > 300
