"""Point location with the face-plane test where the planes' margins matter:
points on vertices, edges and faces and next to them, flattened tetrahedra, far
offsets, extreme scales, cells of no volume.  Against a walk of the same lists
without the planes, bit for bit, and against the oracle's own search."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


CASES = [
    (1.0, 0.0, 1.0), (1.0, 100.0, 1.0), (1.0, 20000.0, 1.0), (1e-6, 0.0, 1.0), (1e7, -3e6, 1.0),
    (1.0, 0.0, 1e-3), (1.0, 1.0, 1e-6), (3e-11, 0.0, 1.0), (1e13, 0.0, 1.0), (1.0, 0.0, 0.0)]


def _points(pos, idx, rng, count):
    """Centres, interior points, vertices, edges and faces of the tetrahedra,
    points within a few roundings of these, and points of the bounds."""
    t = pos[idx.reshape(-1, 4)].astype(np.float64)
    w = rng.dirichlet(np.ones(4), len(t))
    on = [t.mean(1), (w[..., None] * t).sum(1)]
    for k in range(4):
        on.append(t[:, k])
        on.append(0.5 * (t[:, k] + t[:, (k + 1) & 3]))
        on.append(np.delete(t, k, axis=1).mean(1))
        f = rng.dirichlet(np.ones(3), len(t))
        on.append((f[..., None] * np.delete(t, k, axis=1)).sum(1))
    on = np.concatenate(on).astype(np.float32)
    near = on.copy()
    for _ in range(2):
        near = np.nextafter(near, np.where(rng.random(near.shape) < 0.5, -np.inf, np.inf),
                            dtype=np.float32)
    return np.concatenate([on, near, rng.uniform(pos.min(0), pos.max(0), (count, 3))
                           .astype(np.float32)])


def _compare(pkg, oracle, ctx, pos, val, idx, p):
    vrt = pkg.vrt
    f = vrt.DeviceUnstructured(ctx, pos, idx, vertex_data=val)
    dv = vrt.DeviceVolume.from_unstructured(ctx, f, pkg.workloads.albedo_tf(0.8, 64), (0, 1), 1.0)
    o, longest = oracle.tet_walk(pos, val, idx, p)
    assert longest == f.info.max_list
    np.testing.assert_array_equal(vrt.sample_field(ctx, dv, p), o)
    return o


@pytest.mark.parametrize("scale,offset,flat", CASES[:-1])
def test_planes_reject_nothing_that_the_walk_accepts(pkg, oracle, gpu_ctx, scale, offset, flat):
    """Bit for bit the lookups of a walk of the same lists without the planes."""
    pos, val, idx = pkg.vrt.gen_tet_lattice(5, 0.2, 8, 3)
    pos = (pos.astype(np.float64) * scale * np.array([1, 1, flat]) + offset).astype(np.float32)
    p = _points(pos, idx, np.random.default_rng(2), 100000)
    o = _compare(pkg, oracle, gpu_ctx, pos, val, idx, p)
    assert np.isfinite(o).mean() > 0.9


def test_planes_of_a_graded_mesh(pkg, oracle, gpu_ctx):
    """Cells with a handful of entries and one with thousands."""
    pos, val, idx = pkg.vrt.gen_tet_lattice(10, 0.15, 8, 3)
    pos = ((pos + 0.5).clip(1e-6) ** 5).astype(np.float32)
    rng = np.random.default_rng(3)
    p = rng.choice(_points(pos, idx, rng, 20000), 40000, replace=False)
    assert np.isfinite(_compare(pkg, oracle, gpu_ctx, pos, val, idx, p)).mean() > 0.9


@pytest.mark.parametrize("scale,offset,flat", CASES)
def test_sample_on_faces(pkg, oracle, gpu_ctx, scale, offset, flat):
    vrt = pkg.vrt
    pos, val, idx = vrt.gen_tet_lattice(5, 0.2, 8, 3)
    pos = (pos.astype(np.float64) * scale * np.array([1, 1, flat]) + offset).astype(np.float32)
    f = vrt.DeviceUnstructured(gpu_ctx, pos, idx, vertex_data=val)
    tf = pkg.workloads.albedo_tf(0.8, 64)
    dv = vrt.DeviceVolume.from_unstructured(gpu_ctx, f, tf, (0, 1), 1.0)
    ov = oracle.OracleVolume.from_unstructured(pos, idx, tf, (0, 1), 1.0, val)
    rng = np.random.default_rng(1)
    t = pos[idx.reshape(-1, 4)].astype(np.float64)
    w = rng.dirichlet(np.ones(4), len(t))
    on = [t.mean(1), (w[..., None] * t).sum(1)]
    for k in range(4):  # vertices, edges, faces
        on.append(t[:, k])
        on.append(0.5 * (t[:, k] + t[:, (k + 1) & 3]))
        on.append(np.delete(t, k, axis=1).mean(1))
    on = np.concatenate(on)
    lo, hi = pos.min(0), pos.max(0)
    p = np.concatenate([on, rng.uniform(lo, hi, (20000, 3))]).astype(np.float32)
    g, o = vrt.sample_field(gpu_ctx, dv, p), ov.sample(p)
    # a point within rounding of a face may take either side's cell, or fall
    # between the two; no more of them than the general path leaves
    miss = np.isnan(g) != np.isnan(o)
    assert miss.sum() <= max(2, int(2e-3 * len(p))), miss.sum()
    both = ~np.isnan(g) & ~np.isnan(o)
    if flat >= 1e-3 and abs(offset) <= 100.0:
        # inside one tetrahedron: the oracle's own value
        inside = slice(0, 2 * len(t))
        assert not np.isnan(g[inside]).any()
        assert np.mean(g[inside] == o[inside]) >= 0.999
        ok = np.abs(g[both] - o[both]) <= 1e-4
        assert ok.mean() >= 0.999, ok.mean()
