"""Frames smaller and larger than the path tracer's resident waves (claims of
8 to 64 pixels, padding at the right and bottom) hold the same pixels as the
same rows of pixel streams rendered at another schedule."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [(1, 1), (33, 31), (64, 48), (160, 150), (250, 240),
                                          (400, 300), (700, 600)])
def test_sizes_and_schedules(pkg, oracle, gpu_ctx, width, height):
    import dataclasses
    wl = pkg.workloads.cloud_nanovdb_pathtrace(n=64, width=width, height=height, frames=1, brick=8)
    images = []
    for schedule in (1, 2, 3):
        w = dataclasses.replace(wl, params=dict(wl.params, pass_schedule=schedule))
        gs = pkg.workloads.GpuScene(gpu_ctx, w)
        gs.render(0)
        gpu_ctx.sync()
        images.append(gs.frame.color_array().copy())
    np.testing.assert_array_equal(images[0], images[1])
    np.testing.assert_array_equal(images[0], images[2])
    if width * height <= 64 * 48:
        o = oracle.OracleWorkload(wl).pathtrace_frame(0)[0]
        assert oracle.stream_agreement(images[0], o) >= (
            oracle.STREAM_AGREEMENT_MIN if width > 1 else 1.0)
    assert np.isfinite(images[0]).all()
