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


def test_long_lists_where_halves_exceed_the_stack(pkg, oracle, gpu_ctx):
    """Clusters at 2^-i fill the traversal's stack on the way to level 60,
    below which 60,000 triangles are left: the tree with that list as one leaf
    stacks 52 entries, its halves 69 of the 64 that traversals hold."""
    vrt = pkg.vrt
    rng = np.random.default_rng(0)
    s = np.concatenate([np.repeat(2.0 ** -np.arange(110), 14), np.full(60000, 2.0 ** -110)])
    c = s[:, None] * (np.array([1.0, 0, 0]) + 0.2 * rng.random((len(s), 3)))
    tri = (c[:, None] + s[:, None, None] * 0.01 * rng.random((len(s), 3, 3))).astype(np.float32)
    v = tri.reshape(-1, 3)
    mesh = vrt.DeviceMesh(gpu_ctx, v, None, "sah")
    assert mesh.info.stack_bound <= 64 and mesh.info.depth > 69
    scene = vrt.make_scene([], [], [(mesh, (0.7, 0.7, 0.7))])
    r = np.zeros((3000, 8), np.float32)
    k = rng.integers(0, 14 * 40, 3000)  # at triangles of the first 40 scales
    d = rng.normal(size=(3000, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r[:, 3:6] = d
    r[:, :3] = tri[k].mean(1) - 3 * s[k, None] * d
    r[:, 7] = 1e30
    om = oracle.OracleMesh(v, None)
    t, p = vrt.intersect_surfaces(gpu_ctx, scene, r, False)
    to, po = oracle.mesh_intersect(om, r, any_hit=False, brute=True)
    np.testing.assert_array_equal(p, po)
    np.testing.assert_array_equal(t, to)
    assert (po >= 0).mean() > 0.5
    _, pa = vrt.intersect_surfaces(gpu_ctx, scene, r, True)
    np.testing.assert_array_equal(pa >= 0, po >= 0)


def test_long_lists_of_instances(pkg, gpu_ctx):
    """Instance trees hold lists of any length below level 60 as leaves, as the
    instance walk reads whole counts."""
    vrt = pkg.vrt
    rng = np.random.default_rng(1)
    tri = np.array([(-0.5, -0.5, 0), (0.5, -0.5, 0), (0, 0.5, 0)], np.float32)
    mesh = vrt.DeviceMesh(gpu_ctx, tri, None, "sah")
    s = np.concatenate([2.0 ** -np.arange(90), np.full(400, 2.0 ** -90)])
    xf = np.zeros((len(s), 3, 4), np.float32)
    xf[:, [0, 1, 2], [0, 1, 2]] = 0.05
    xf[:, 0, 3] = s * (1 + 0.2 * rng.random(len(s)))
    tls = vrt.DeviceTls(gpu_ctx, [(mesh, x, (0.7, 0.7, 0.7)) for x in xf])
    assert tls.info.stack_bound <= 8
    scene = vrt.make_scene([], [], [], tls=tls)
    r = np.zeros((600, 8), np.float32)
    r[:, 0] = rng.uniform(-0.1, 1.3, 600)
    r[:, 1] = rng.uniform(-0.03, 0.03, 600)
    r[:, 2], r[:, 5], r[:, 7] = 1.0, -1.0, 1e30
    _, p = vrt.intersect_surfaces(gpu_ctx, scene, r, True)
    x = (r[:, None, 0] - xf[None, :, 0, 3]) / 0.05
    y = r[:, None, 1] / 0.05
    margin = np.minimum(y + 0.5, 0.5 - y - 2 * np.abs(x)).max(1)  # > 0: inside one
    clear = np.abs(margin) > 1e-3
    np.testing.assert_array_equal(p[clear] >= 0, margin[clear] > 0)
    assert 50 < (margin > 0).sum() < 550
