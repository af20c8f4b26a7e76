"""The binned splat at the edges of its lists, regions and jobs, bit for bit
against the point-parallel splat (which the oracle's frames pin)."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
from helpers import assert_same, flush

pytestmark = pytest.mark.gpu


def _frames(gpu, arrays, w, h, ss, spp, eye, modes, gpb=0, **kw):
    st = gpu.RenderSettings(w, h, spp, ss, gaussians_per_block=gpb)
    f = gpu.frame_params(eye, (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=ss, frame=3, spp=spp, background=(0.2, 0.4, 0.6),
                         **kw)
    out = []
    for mode in modes:
        flush(f"{w}x{h} ss {ss} spp {spp} n {arrays.n} mode {mode}")
        r = H.GpuRunner(arrays, st)
        r.p.set_splat_mode(mode)
        out.append(r.render(f, [gpu.DBG_FRAMEBUFFER]))
    return out


def _same(gpu, a, b, what):
    assert_same(f"{what} fb", a.debug[gpu.DBG_FRAMEBUFFER], b.debug[gpu.DBG_FRAMEBUFFER])
    assert_same(f"{what} colour", a.color, b.color)
    assert_same(f"{what} depth", a.depth, b.depth)


# one pixel, a region less one pixel, a region, a region and one pixel, ragged tiles
@pytest.mark.parametrize("spp", [1, 2, 3, 4])
@pytest.mark.parametrize("size", [(1, 1), (127, 63), (128, 64), (129, 65), (333, 190)])
def test_binned_region_edges(gpu, size, spp):
    """Regions cut by the screen, regions without a point (cleared with the
    lists) and regions of one and of several jobs."""
    w, h = size
    arrays = H.scene(0x5EED0801 + spp, 9_000, dict(H.C1, half_extent=4.0, log_scale_mu=-2.5)).morton_sorted()
    a, b = _frames(gpu, arrays, w, h, 1, spp, (0.0, 3.0, -25.0), (gpu.Pass.SPLAT_BINNED, gpu.Pass.SPLAT_POINT_PARALLEL))
    assert a.stats["splat_binned"] == 1 and a.stats["splat_fallback"] == 0, a.stats
    _same(gpu, a, b, f"{size} spp {spp}")


@pytest.mark.parametrize("n", [1, 2, 63, 4097])
def test_binned_big_gaussians(gpu, n):
    """Gaussians over more than four regions (their points in slices of 1024,
    splatted after the regions), alone and beside small ones."""
    arrays = H.scene(0x5EED0811, n, dict(H.C1, half_extent=3.0, log_scale_mu=-3.0)).morton_sorted()
    k = max(1, n // 50)
    arrays.scales[:k] = np.float32(1.5)
    arrays.opacities[:k] = np.float32(0.7)
    a, b = _frames(gpu, arrays, 640, 360, 2, 4, (0.0, 1.0, -9.0), (gpu.Pass.SPLAT_BINNED, gpu.Pass.SPLAT_POINT_PARALLEL))
    assert a.stats["splat_fallback"] == 0 and a.stats["bin_big"] >= 1, a.stats
    assert a.stats["num_points"][0] > 1024
    _same(gpu, a, b, f"{n} Gaussians")


@pytest.mark.parametrize("spp", [1, 4])
def test_binned_long_gaussians(gpu, spp):
    """Gaussians in few regions with more points than one wave should list
    (16384; a frame of 240 x 240 pixels allows one 28800)."""
    arrays = H.scene(0x5EED0841, 2000, dict(H.C1, half_extent=3.0, log_scale_mu=-3.0)).morton_sorted()
    arrays.scales[::500] = np.float32(40.0)
    arrays.opacities[::500] = np.float32(0.9)
    a, b = _frames(gpu, arrays, 240, 240, 1, spp, (0.0, 1.0, -9.0), (gpu.Pass.SPLAT_BINNED, gpu.Pass.SPLAT_POINT_PARALLEL))
    assert a.stats["splat_fallback"] == 0 and a.stats["num_points"][0] > 4 * 16384, a.stats
    assert (a.stats["bin_big"] >= 4) if spp < 3 else (a.stats["bin_big"] >= 1), a.stats
    _same(gpu, a, b, f"spp {spp}")


@pytest.mark.parametrize("n", [30_000, 90_000, 190_000, 400_000])
def test_binned_batch_list_steps(gpu, n):
    """Lists written in steps of 1, 2, 4 and 8 entries a thread (16 views share
    the workgroups: 65536 threads each), ragged at the end."""
    w, h, v = 160, 90, 16
    arrays = H.scene(0x5EED0851, n + 37, dict(H.C1, half_extent=6.0, log_scale_mu=-3.0))
    scene, stream = gpu.Scene(arrays), gpu.Stream()
    frames = [gpu.frame_params((0.1 * i, 1.0, -22.0), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=2, frame=2 + i, spp=2)
              for i in range(v)]
    out = [(gpu.DeviceArray((h, w, 3), np.float32, zero=True), gpu.DeviceArray((h, w), np.float32, zero=True))
           for _ in range(v)]
    got = []
    for mode in (gpu.Pass.SPLAT_BINNED, gpu.Pass.SPLAT_POINT_PARALLEL):
        flush(f"list steps n {n} mode {mode}")
        b = gpu.Batch(scene, v, w, h, 2, 2)
        b.set_splat_mode(mode)
        b.render(frames, [c for c, _ in out], [d for _, d in out], stream)
        stats = b.view_stats(0, stream)
        assert stats["splat_binned"] == (mode == gpu.Pass.SPLAT_BINNED) and stats["splat_fallback"] == 0, stats
        got.append([(c.download(), d.download()) for c, d in out])
        b.close()
    for i, (x, y) in enumerate(zip(*got)):
        assert_same(f"view {i} colour", x[0], y[0])
        assert_same(f"view {i} depth", x[1], y[1])


@pytest.mark.parametrize("spp", [1, 4])
def test_binned_list_overflow(gpu, spp):
    """More listed points than a forced list holds (twice the budget): every
    Gaussian lies on the corner of four regions, so each point is listed four
    times.  The frame is splatted point-parallel from a cleared framebuffer,
    and the next frame on the same pass is binned."""
    arrays = H.scene(0x5EED0881, 4000, dict(H.C1, half_extent=0.05, log_scale_mu=-1.6, log_scale_sigma=0.1))
    w = 256 if spp == 1 else 128
    st = gpu.RenderSettings(w, w, spp, 1, max_number_of_points=1 << 20, fully_disable_hierarchical_culling=True)
    a, b = H.GpuRunner(arrays, st), H.GpuRunner(arrays, st)
    a.p.set_splat_mode(gpu.Pass.SPLAT_BINNED)
    b.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    fallbacks = []
    for k, z in enumerate((-4.0, -60.0, -4.0, -60.0)):
        flush(f"list overflow spp {spp} frame {k}")
        f = gpu.frame_params((0.0, 0.0, z), (0, 0, 0), (0, 1, 0), 45.0, w, w, ss=1, frame=1 + k, spp=spp,
                             background=(0.2, 0.4, 0.6))
        x, y = (r.render(f, [gpu.DBG_FRAMEBUFFER]) for r in (a, b))
        _same(gpu, x, y, f"spp {spp} frame {k}")
        assert x.stats["splat_binned"] == 1
        fallbacks.append(x.stats["splat_fallback"])
    assert fallbacks == [1, 0, 1, 0], fallbacks


def test_binned_without_bounds(gpu):
    """A scene of more than half as many Gaussians as points can be binned,
    most of them out of view: no bounds are written, the lists read them from
    the records.  Single passes and a batch."""
    w, h = 320, 180
    arrays = H.scene(0x5EED0891, 600_000, dict(H.C1, half_extent=60.0, log_scale_mu=-3.0)).morton_sorted()
    st = gpu.RenderSettings(w, h, 2, 2)
    f = gpu.frame_params((0.0, 1.0, -5.0), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=2, frame=3, spp=2, hierarchical=True,
                         background=(0.2, 0.4, 0.6))
    a, b = H.GpuRunner(arrays, st), H.GpuRunner(arrays, st)
    b.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    flush("no bounds: single pass")
    x, y = (r.render(f, [gpu.DBG_FRAMEBUFFER]) for r in (a, b))
    assert 2 * arrays.n > 8 * w * h >= x.stats["num_points"][0] > 50_000, x.stats
    assert x.stats["splat_binned"] == 1 and x.stats["splat_fallback"] == 0, x.stats
    _same(gpu, x, y, "no bounds")
    flush("no bounds: batch")
    batch = gpu.Batch(a.scene, 1, w, h, 2, 2)
    batch.render([f], [a.color], [a.depth], a.stream)
    stats = batch.view_stats(0, a.stream)
    assert stats["splat_binned"] == 1 and stats["splat_fallback"] == 0, stats
    assert_same("batch colour", a.color.download(), y.color)
    assert_same("batch depth", a.depth.download(), y.depth)
    batch.close()


def _auto_frames(gpu, arrays, w, h, spp, eyes, ss=2, **kw):
    """The automatic choice's statistics per frame, its images checked against
    the point-parallel splat's."""
    st = gpu.RenderSettings(w, h, spp, ss, fully_disable_hierarchical_culling=True)
    a, b = H.GpuRunner(arrays, st), H.GpuRunner(arrays, st)
    b.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    out = []
    for k, eye in enumerate(eyes):
        flush(f"automatic {w}x{h} n {arrays.n} frame {k}")
        f = gpu.frame_params(eye, (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=ss, frame=3 + k, spp=spp,
                             background=(0.2, 0.4, 0.6), **kw)
        x, y = (r.render(f, [gpu.DBG_FRAMEBUFFER]) for r in (a, b))
        _same(gpu, x, y, f"{w}x{h} n {arrays.n} frame {k}")
        out.append((x.stats["splat_binned"], x.stats["splat_fallback"]))
    return out


def test_binned_auto_large_framebuffer(gpu):
    """Points of 4 samples from 6 * 2^20 framebuffer words on: binned with at
    least 3e13 / words points (4.6M here), else stood down on the device, frame
    by frame; not tried in smaller framebuffers or scenes, nor where occluded
    Gaussians are culled from a scene of fewer Gaussians than that."""
    cfg = dict(H.C1, half_extent=8.0)
    arrays = H.scene(0x5EED0821, 950_000, cfg).morton_sorted()
    near, far = (0.0, 3.0, -25.0), (0.0, 3.0, -60.0)
    assert _auto_frames(gpu, arrays, 1700, 956, 1, [near, far, near]) == [(1, 0), (1, 3), (1, 0)]
    assert _auto_frames(gpu, arrays, 1400, 780, 1, [near]) == [(0, 0)]
    assert _auto_frames(gpu, arrays, 1700, 956, 1, [near, near], occlusion=True) == [(0, 0)] * 2
    assert _auto_frames(gpu, H.scene(0x5EED0821, 400_000, cfg), 1700, 956, 1, [near]) == [(0, 0)]


@pytest.mark.parametrize("n,size,views,binned", [(900_000, (1280, 720), 1, 1), (400_000, (1280, 720), 1, 0),
                                                 (400_000, (1280, 720), 3, 1), (200_000, (1280, 720), 9, 0),
                                                 (900_000, (480, 270), 9, 0)])
def test_binned_auto_batch(gpu, n, size, views, binned):
    """Views of points of 4 samples: more than 2^20 words, a Gaussian per 16 of
    them, Gaussians * words * views >= 3e12."""
    w, h = size
    arrays = H.scene(0x5EED0871, n, dict(H.C1, half_extent=8.0, log_scale_mu=-4.5))
    scene, stream = gpu.Scene(arrays), gpu.Stream()
    f = [gpu.frame_params((0.0, 3.0, -25.0 - i), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=2, frame=3, spp=1)
         for i in range(views)]
    out = [(gpu.DeviceArray((h, w, 3), np.float32, zero=True), gpu.DeviceArray((h, w), np.float32, zero=True)) for _ in f]
    flush(f"automatic batch {size} n {n} views {views}")
    got = []
    for mode in (gpu.Pass.SPLAT_AUTO, gpu.Pass.SPLAT_POINT_PARALLEL):
        b = gpu.Batch(scene, views, w, h, 1, 2)
        b.set_splat_mode(mode)
        b.render(f, [c for c, _ in out], [d for _, d in out], stream)
        for i in range(views):
            stats = b.view_stats(i, stream)
            assert stats["splat_fallback"] == 0 and stats["splat_binned"] == (binned if mode == 0 else 0), (i, stats)
        got.append([(c.download(), d.download()) for c, d in out])
        b.close()
    for i, (x, y) in enumerate(zip(*got)):
        assert_same(f"view {i} colour", x[0], y[0])
        assert_same(f"view {i} depth", x[1], y[1])


def test_binned_auto_dense_large_framebuffer(gpu):
    """Points of 9 samples: up to 8 samples per word, in framebuffers of more
    than 2^22 words up to 6 for every 2^22 words (20 here)."""
    arrays = H.scene(0x5EED0861, 2_700_000, dict(H.C1, half_extent=5.0, log_scale_mu=-4.2)).morton_sorted()
    far, mid, near = ((0.0, 3.0, d) for d in (-40.0, -19.0, -9.5))
    assert _auto_frames(gpu, arrays, 640, 360, 1, [far], ss=3) == [(1, 2)]  # 15 samples per word
    assert _auto_frames(gpu, arrays, 1700, 956, 1, [mid, near], ss=3) == [(1, 0), (1, 2)]  # 9.8 and 27


def test_first_culled_frame_is_point_parallel(gpu):
    """4 samples a point in a scene that may be too dense to bin: the first
    frame with occlusion culling, which nothing culls, takes no lists; later
    ones do.  The same images as point-parallel throughout."""
    arrays = H.scene(0x5EED0831, 7_400_000, dict(H.C1, half_extent=30.0, log_scale_mu=-4.0))
    w, h = 1700, 956
    st = gpu.RenderSettings(w, h, 1, 2, gaussians_per_block=256)
    a, b = H.GpuRunner(arrays, st), H.GpuRunner(arrays, st)
    b.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    for k in range(3):
        f = gpu.frame_params((0.1 * k, 3.0, -20.0), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=2, frame=k + 1,
                             occlusion=True, hierarchical=True, background=(0.2, 0.4, 0.6))
        flush(f"first culled frame: frame {k}")
        x, y = (r.render(f, [gpu.DBG_FRAMEBUFFER]) for r in (a, b))
        assert x.stats["splat_binned"] == (0 if k == 0 else 1), (k, x.stats)
        _same(gpu, x, y, f"frame {k}")


def test_captured_first_culled_frame(gpu):
    """... but not when the caller captures it: its replays are no first frames."""
    arrays = H.scene(0x5EED0831, 7_400_000, dict(H.C1, half_extent=30.0, log_scale_mu=-4.0))
    w, h = 1700, 956
    st = gpu.RenderSettings(w, h, 1, 2, gaussians_per_block=256)
    a, b = H.GpuRunner(arrays, st), H.GpuRunner(arrays, st)
    b.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    f = gpu.frame_params((0.1, 3.0, -20.0), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=2, frame=1, occlusion=True,
                         hierarchical=True, background=(0.2, 0.4, 0.6))
    hip, stream = gpu.lib, a.stream.handle
    graph, exe = C.c_void_p(), C.c_void_p()
    flush("captured first culled frame")
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread local
    a.p.render(f, a.color, a.depth, a.stream)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    for k in range(3):
        flush(f"captured first culled frame: replay {k}")
        assert hip.hipGraphLaunch(exe, stream) == 0
        a.stream.synchronize()
        assert a.p.stats(a.stream)["splat_binned"] == 1
        want = b.render(f)
        assert np.array_equal(a.color.download(), want.color) and np.array_equal(a.depth.download(), want.depth), k
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
