"""The resolves at the edges of their tiles and vectors, and on images off
the vectors' boundaries, against the oracle bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import assert_same, flush

pytestmark = pytest.mark.gpu


class _At:
    """A device array at `off` elements into its allocation."""

    def __init__(self, gpu, a, off):
        self.base = gpu.DeviceArray((a.size + off,), a.dtype, zero=True)
        self.a, self.off = a, off
        self.ptr = C.c_void_p(self.base.ptr.value + off * a.itemsize)
        self.upload(a)

    def upload(self, a):
        self.base.upload(np.concatenate([np.zeros(self.off, a.dtype), a.reshape(-1)]))

    def download(self):
        return self.base.download()[self.off:].reshape(self.a.shape)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("size", [(1, 1), (3, 2), (63, 15), (64, 16), (65, 17), (130, 33), (320, 49)])
def test_resolve_sizes(gpu, size, off):
    import orc
    w, h = size
    rng = np.random.default_rng(w * 1000 + h)
    cur = rng.uniform(-0.1, 1.2, (h, w, 3)).astype(np.float32)
    prev = rng.uniform(0.0, 1.0, (h, w, 3)).astype(np.float32)
    dep = rng.uniform(0.9, 1.0, (h, w)).astype(np.float32)
    cur[0, 0, 0], prev[-1, -1, 2] = np.nan, np.inf
    proj = gpu.perspective(45.0, w / h, 0.2, 1e4)
    M = gpu.taa_reprojection(gpu.mat4_mul(proj, gpu.look_at((0.0, 0.0, -30.0), (0.0, 0.0, 0.0))),
                             gpu.look_at((0.1, 0.05, -30.0), (0.0, 0.0, 0.0)), proj)
    dc, dp, dd = (_At(gpu, a, off) for a in (cur, prev, dep))
    out, rgb = _At(gpu, np.zeros_like(cur), off), _At(gpu, np.zeros(cur.shape, np.uint8), off)
    flush(f"resolve {size} offset {off}")
    for fn in (0, 3):
        gpu.resolve_taa(dc, dd, dp, dd, M, 0.9, w, h, fn, out, rgb)
        c, r = orc.resolve_taa(cur, dep, prev, dep, M, 0.9, w, h, fn)
        ok = np.isfinite(c)
        assert np.array_equal(np.isfinite(out.download()), ok)
        assert_same(f"taa {fn}", out.download()[ok], c[ok])
        assert_same(f"taa rgb {fn}", rgb.download()[ok], r[ok])
    cur[0, 0, 0], prev[-1, -1, 2] = 0.25, 0.5
    for n in (1, 2):
        dc.upload(cur)
        dp.upload(prev)
        gpu.resolve_progressive(dc, dp, w, h, n, rgb)
        c, a, r = orc.resolve_progressive(cur, prev, w, h, n)
        assert_same(f"progressive {n}", dc.download(), c)
        assert_same(f"accum {n}", dp.download(), a)
        assert_same(f"progressive rgb {n}", rgb.download(), r)
