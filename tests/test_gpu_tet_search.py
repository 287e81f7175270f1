"""Point location with the face-plane test against the oracle's search where
the planes' margins matter: points on vertices, edges and faces, flattened
tetrahedra, far offsets, extreme scales and cells of no volume."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale,offset,flat", [
    (1.0, 0.0, 1.0), (1.0, 100.0, 1.0), (1.0, 20000.0, 1.0), (1e-6, 0.0, 1.0), (1e7, -3e6, 1.0),
    (1.0, 0.0, 1e-3), (1.0, 1.0, 1e-6), (3e-11, 0.0, 1.0), (1e13, 0.0, 1.0), (1.0, 0.0, 0.0)])
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
