"""What a pass allocates for the binned splat: nothing where no frame of its
settings can be binned, as much as the estimate says elsewhere, and no more
than a server's budget leaves room for."""
import ctypes as C

import numpy as np
import pytest

import helpers as H
from helpers import assert_same, flush

pytestmark = pytest.mark.gpu


def _estimate(gpu, st, scene):
    s = st.c()
    return int(gpu.lib.gps_pass_estimate_bytes(C.byref(s), scene.handle))


def _device_bytes(gpu, p):
    return int(gpu.lib.gps_pass_device_bytes(p.handle))


def _frame(gpu, w, h, ss, spp, **kw):
    return gpu.frame_params((0.0, 3.0, -25.0), (0, 0, 0), (0, 1, 0), 45.0, w, h, ss=ss, spp=spp, frame=3,
                            background=(0.2, 0.4, 0.6), **kw)


@pytest.fixture(scope="module")
def small(gpu):
    return H.scene(0x5EED0B01, 100_000, dict(H.C1, half_extent=6.0)).morton_sorted()


# width, height, ss, spp, flexible size; whether a frame can be binned automatically
@pytest.mark.parametrize("w,h,ss,spp,flexible,binnable", [
    (3840, 2160, 1, 1, False, False),   # one sample per point
    (1280, 720, 2, 1, False, False),    # four samples, not a large framebuffer
    (3840, 2160, 1, 3, True, False),
    (640, 360, 1, 4, False, False),
    (640, 360, 2, 5, False, False),     # more layers than the binned splat has
    (640, 360, 2, 5, True, True),       # ... but smaller frames may have fewer
    (640, 360, 2, 2, False, True),
    (640, 360, 3, 1, False, True),
    (1, 1, 3, 4, False, True),
])
def test_pass_bytes(gpu, small, w, h, ss, spp, flexible, binnable):
    scene = gpu.Scene(small)
    st = gpu.RenderSettings(w, h, spp, ss, flexible_frame_size=flexible)
    n, px = small.n, w * h
    fb = 2 * 8 * ((w * ss + 63) // 64 * 64) * ((h * ss + 63) // 64 * 64) * spp
    p = gpu.Pass(st, scene)
    have = _device_bytes(gpu, p)
    print(f"{w}x{h} ss {ss} spp {spp}: {have} bytes, framebuffers {fb}", flush=True)
    assert have == _estimate(gpu, st, scene)
    # records, lists and masks of the scene, the chunk tables of the budget, Hi-Z
    others = fb + 100 * n + 8 * px + (8 << 20)
    if binnable:
        assert have <= others + 16 * n + 8 * 16 * px + (4 << 20)
    else:
        assert have <= others
    p.close()
    scene.close()


def test_estimate_follows_the_budget(gpu, small):
    scene = gpu.Scene(small)
    by = [_estimate(gpu, gpu.RenderSettings(1920, 1080, 2, 2, max_number_of_points=b), scene)
          for b in (1 << 20, 1 << 22, 1 << 24, 1 << 28)]
    assert by[1] - by[0] > 8 * 2 * 3 * (1 << 20) and by[0] < by[1] < by[2] < by[3]
    assert by[3] - by[2] < 16 << 20  # the frame's own 16 points per pixel hold here


@pytest.mark.parametrize("w,h,binnable,not_binnable", [
    (3840, 2160, 3840 * 2160 // 4, 3840 * 2160 // 4 - 1),      # a Gaussian per 16 words
    (1700, 956, 16 * 1700 * 956, 16 * 1700 * 956 + 1),         # 4 Gaussians per word
    (1666, 944, None, 20_000_000),                             # 6 * 2^20 words
    (1668, 944, 20_000_000, None),
])
def test_ends_of_the_rule_for_points_of_four_samples(gpu, w, h, binnable, not_binnable):
    """The estimate counts a list exactly where such a frame may be binned
    (the scenes hold no data)."""
    st = gpu.RenderSettings(w, h, 1, 2, max_number_of_points=1 << 26, fully_disable_hierarchical_culling=True)
    for n, can in ((binnable, True), (not_binnable, False)):
        if n is None:
            continue
        handle = C.c_void_p()
        assert gpu.lib.gps_scene_create_empty(n, 0, gpu.FORMAT_HALF_FP8, C.byref(handle)) == 0
        settings = st.c()
        bytes_ = int(gpu.lib.gps_pass_estimate_bytes(C.byref(settings), handle))
        gpu.lib.gps_scene_destroy(handle)
        fb = 2 * 8 * ((w * 2 + 63) // 64 * 64) * ((h * 2 + 63) // 64 * 64)
        others = fb + 78 * n + 8 * w * h + (8 << 20)
        print(f"{w}x{h} n {n}: {bytes_} bytes, {others} without lists", flush=True)
        assert (bytes_ > others + 16 * n) if can else (bytes_ < others + 4 * n), (n, bytes_, others)


def test_supersampling_that_can_be_binned_later(gpu, small):
    """A pass made for frames that cannot be binned takes its list with the
    framebuffers of the first frame that can."""
    w, h = 333, 190
    st = gpu.RenderSettings(w, h, 2, 1)
    r = H.GpuRunner(small, st)
    sizes = [_device_bytes(gpu, r.p)]
    for ss in (1, 2, 3, 2, 1):
        f = _frame(gpu, w, h, ss, 2)
        flush(f"supersampling {ss}")
        r.p.set_splat_mode(gpu.Pass.SPLAT_AUTO)
        a = r.render(f, [gpu.DBG_FRAMEBUFFER])
        r.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
        b = r.render(f, [gpu.DBG_FRAMEBUFFER])
        assert a.stats["splat_binned"] == (1 if ss > 1 else 0) and a.stats["splat_fallback"] == 0, (ss, a.stats)
        assert_same(f"ss {ss} framebuffer", a.debug[gpu.DBG_FRAMEBUFFER], b.debug[gpu.DBG_FRAMEBUFFER])
        assert_same(f"ss {ss} colour", a.color, b.color)
        sizes.append(_device_bytes(gpu, r.p))
    fb = [2 * 8 * 2 * ((w * ss + 63) // 64 * 64) * ((h * ss + 63) // 64 * 64) for ss in (1, 1, 2, 3, 2, 1)]
    lists = [s - f for s, f in zip(sizes, fb)]
    assert lists[0] == lists[1] < lists[2], (sizes, fb)


def _captured(gpu, r, frame):
    """The frame captured by its caller: graph and executable."""
    hip, st = gpu.lib, r.stream.handle
    graph, exe = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(st, 1) == 0  # thread local
    r.p.render(frame, r.color, r.depth, r.stream)
    assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    return graph, exe


def test_captured_frame_of_another_supersampling(gpu, small):
    """Framebuffers this small do not change with the factor: a frame that the
    caller captures takes no list either, the next eager one does."""
    w, h = 16, 12
    st = gpu.RenderSettings(w, h, 1, 1)
    r, other = H.GpuRunner(small, st), H.GpuRunner(small, st)
    first, third = (_frame(gpu, w, h, ss, 1) for ss in (1, 3))
    flush("captured supersampling: eager frames")
    r.render(first)
    other.p.set_splat_mode(gpu.Pass.SPLAT_POINT_PARALLEL)
    want, again = other.render(third), other.render(first)
    before = _device_bytes(gpu, r.p)
    graph, exe = _captured(gpu, r, third)
    assert _device_bytes(gpu, r.p) == before
    for k in range(3):
        flush(f"captured supersampling: replay {k}")
        assert gpu.lib.hipGraphLaunch(exe, r.stream.handle) == 0
        r.stream.synchronize()
        assert_same(f"replay {k} colour", r.color.download(), want.color)
        assert_same(f"replay {k} depth", r.depth.download(), want.depth)
        assert_same(f"eager {k}", r.render(first).color, again.color)
    got = r.render(third)
    assert got.stats["splat_binned"] == 1, got.stats  # though too dense for the lists
    assert _device_bytes(gpu, r.p) > before
    assert_same("eager colour", got.color, want.color)
    assert gpu.lib.hipGraphExecDestroy(exe) == 0 and gpu.lib.hipGraphDestroy(graph) == 0


def test_forced_binning_allocates_once(gpu, small):
    scene = gpu.Scene(small)
    st = gpu.RenderSettings(640, 360, 1, 1, max_number_of_points=2_000_000)
    p = gpu.Pass(st, scene)
    before = _device_bytes(gpu, p)
    p.set_splat_mode(gpu.Pass.SPLAT_BINNED)
    forced = _device_bytes(gpu, p)
    assert 8 * 4_000_000 <= forced - before <= 8 * 4_000_000 + 16 * small.n + (2 << 20)
    p.set_splat_mode(gpu.Pass.SPLAT_AUTO)
    p.set_splat_mode(gpu.Pass.SPLAT_BINNED)
    assert _device_bytes(gpu, p) == forced
    p.close()


def test_server_budget_without_room_for_full_lists(gpu, small):
    """Two slots and two scenes: a budget short of the full lists by three
    quarters holds every pass, with shorter ones, and the same images."""
    w, h = 640, 360
    other = H.scene(0x5EED0B02, 300_000, dict(H.C1, half_extent=6.0)).morton_sorted()
    scenes = [gpu.Scene(small), gpu.Scene(other)]
    st = gpu.RenderSettings(w, h, 4, 2, flexible_frame_size=True)
    full = [_estimate(gpu, st, s) for s in scenes]
    lists = 2 * 2 * 8 * 16 * w * h  # of all four passes, at least
    frames = [_frame(gpu, 333 + 50 * i, 190 + 20 * i, 2, 4, hierarchical=True) for i in range(4)]

    def run(budget):
        srv = gpu.Server(slots=2, max_width=w, max_height=h, max_spp=4, max_supersampling=2, hbm_budget_bytes=budget)
        ids = [srv.add_scene(s) for s in scenes]
        srv.prepare()
        out = []
        srv.start()
        for i, f in enumerate(frames):
            img = np.zeros((f.height, f.width, 3), np.float32)
            srv.submit(ids[i % 2], f, -1.0, None, img)
            out.append(img)
        srv.drain(120_000)
        done = srv.poll(64)
        stats = srv.stats()
        srv.close()
        assert len(done) == 4 and all(d["status"] == 0 for d in done)
        return out, stats

    flush("server with room for everything")
    a, sa = run(0)
    need = sa["hbm_used_bytes"]
    assert sa["passes_created"] == 4 and need >= 2 * sum(full)
    flush("server with a quarter of the lists' room")
    b, sb = run(need - lists * 3 // 4)
    print(sa, sb)
    assert sb["passes_created"] == 4 and sb["passes_evicted"] == 0
    assert sb["hbm_used_bytes"] <= need - lists * 3 // 4
    for i, (x, y) in enumerate(zip(a, b)):
        assert_same(f"request {i}", x, y)
