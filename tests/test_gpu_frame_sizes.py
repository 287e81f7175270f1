"""Frames smaller and larger than the path tracer's resident waves (first units
of 8 to 64 pixels, later claims of 16 to 64, padding at the right and bottom):
the same pixels at every schedule, each pixel written once, and the oracle's
image."""
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
        gs.frame.color.upload(np.full(width * height * 4, np.nan, np.float32))
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


def _workload(wls, scene, width, height):
    kw = dict(width=width, height=height, frames=1)
    if scene == "cloud":
        return wls.cloud_nanovdb_pathtrace(n=64, brick=8, **kw)
    if scene == "tets":
        return wls.tets_pathtrace(n=8, grid=16, **kw)
    if scene == "mixed":
        return wls.mixed_pathtrace(level=3, vol_n=32, **kw)
    if scene == "instances":
        return wls.instanced_pathtrace(**kw)
    wl = wls.fbm_pathtrace(n=32, brick=8, max_bounce=0 if scene == "cache" else 8, **kw)
    wl.params["ratio_tracking"] = scene == "ratio"
    return wl


@pytest.mark.parametrize("scene", ["fbm", "ratio", "cloud", "tets", "mixed", "instances", "cache"])
@pytest.mark.parametrize("width,height", [(250, 241), (400, 300), (701, 599)])
def test_every_pixel_once_against_the_oracle(pkg, oracle, gpu_ctx, scene, width, height):
    """Units claimed from the queues' counters as well as those by position, for
    each size of claim.  "cache": a cache of zero weights, whose frame is that
    of paths cut at their first vertex."""
    vrt, wls = pkg.vrt, pkg.workloads
    wl = _workload(wls, scene, width, height)
    gs = wls.GpuScene(gpu_ctx, wl, accum64=True,
                      params=dict(max_bounce=8) if scene == "cache" else None)
    gs.frame.reset()
    gs.frame.color.upload(np.full(width * height * 4, np.nan, np.float32))
    if scene == "cache":
        nrc = vrt.Nrc(gpu_ctx)
        try:
            nrc.set_params(np.zeros(nrc.nparams, np.float32))
            gs.render_nrc(nrc, gs.nrc_options(train=False), 0)
            gpu_ctx.sync()
        finally:
            nrc.close()
    else:
        gs.render(0)
        gpu_ctx.sync()
    image = gs.frame.color_array()
    assert np.isfinite(image).all()
    # the running sums: written twice they would hold twice the sample
    np.testing.assert_array_equal(gs.frame.accum64_array(), image.astype(np.float64))
    assert (image[..., 3] > 0).all()
    o = oracle.OracleWorkload(wl).pathtrace_frame(0)[0]
    same = np.all(np.abs(image - o) <= 1e-4 * np.maximum(1, np.abs(o)), -1)
    assert same.mean() >= oracle.STREAM_AGREEMENT_MIN
    # no unit is missing or misplaced: a rounding that decides a collision
    # differently strikes single pixels (1 in 10^3 to 10^4), not most of a tile
    pad = np.pad(same, ((0, -height % 8), (0, -width % 8)), constant_values=True)
    tiles = pad.reshape(pad.shape[0] // 8, 8, pad.shape[1] // 8, 8).mean((1, 3))
    assert tiles.min() >= 0.5, tiles.min()
