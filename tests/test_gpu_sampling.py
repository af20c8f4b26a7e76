"""The splat's sampling transform as the device compiles it (hardware root,
conversion and clamps) against the general functions it stands for, bit for
bit; zeros count as equal whatever their sign."""
import ctypes as C

import numpy as np
import pytest

from helpers import flush

pytestmark = pytest.mark.gpu


def _run(gpu, kind, words, n=None):
    words = np.ascontiguousarray(words, np.uint32)
    n = words.size if n is None else n
    d_in, d_out = gpu.DeviceArray(words.shape, np.uint32), gpu.DeviceArray((n,), np.uint32)
    d_in.upload(words)
    flush(f"sampling kind {kind}: {n} inputs")
    gpu.check(gpu.lib.gps_selftest_sampling(kind, d_in.ptr, d_out.ptr, n, None), "selftest")
    return d_out.download()


def _math(gpu, kind, x):
    d_in, d_out = gpu.DeviceArray(x.shape, np.float32), gpu.DeviceArray(x.shape, np.float32)
    d_in.upload(x)
    gpu.check(gpu.lib.gps_selftest_math(kind, d_in.ptr, d_out.ptr, x.size, None), "selftest")
    return d_out.download()


def _same_floats(got, want):
    got = got.view(np.float32)
    assert not np.isnan(got).any()
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, (bad.size, bad[:4], got[bad[:4]], want[bad[:4]])


def test_radius_root(gpu):
    """Every float in [1, 4) (scaling by 4 commutes), samples from 2^-100 to
    2^64, every 5th float of the radius' range, and both zeros."""
    one = np.arange(1 << 24, dtype=np.uint32) + np.uint32(0x3F800000)
    rng = np.random.default_rng(1)
    wide = np.exp2(rng.uniform(-100.0, 64.0, 1 << 20)).astype(np.float32)
    wide = wide[wide < 2.0 ** 64].view(np.uint32)
    lo, hi = (int(np.float32(v).view(np.uint32)) for v in (2.0 ** -24, 171.0))
    radius = np.arange(lo, hi, 5, dtype=np.int64).astype(np.uint32)
    zeros = np.array([0, 0x80000000], np.uint32)
    for part in (one, wide, radius, zeros):
        _same_floats(_run(gpu, 0, part), np.sqrt(np.abs(part.view(np.float32))))


def test_saturating_conversion(gpu):
    rng = np.random.default_rng(2)
    x = np.concatenate([rng.uniform(-70000, 70000, 1 << 18), rng.uniform(-3e9, 3e9, 1 << 18),
                        [0.0, -0.0, 0.99999994, -0.99999994, 2147483520.0, 2147483648.0, -2147483648.0, -2147483904.0,
                         1e30, -1e30, np.inf, -np.inf, np.nan, 1e-40]]).astype(np.float32)
    want = np.where(np.isnan(x), 0.0, np.clip(np.trunc(x.astype(np.float64)), -2.0 ** 31, 2.0 ** 31 - 1)).astype(np.int64)
    assert np.array_equal(_run(gpu, 1, x.view(np.uint32)).view(np.int32), want)


def test_log(gpu):
    """Every float in [1/4, 1] and samples down to 1e-37, against the general
    logarithm (which the oracle pins)."""
    one = np.arange(0x3E800000, 0x3F800001, dtype=np.uint32).view(np.float32)
    rng = np.random.default_rng(3)
    small = np.exp(rng.uniform(np.log(1e-37), 0.0, 1 << 21)).astype(np.float32)
    for part in (one, small[small >= np.float32(1e-37)]):
        _same_floats(_run(gpu, 2, part.view(np.uint32)), np.float32(-2.0) * _math(gpu, 1, np.ascontiguousarray(part)))


@pytest.mark.parametrize("kind,general", [(3, 2), (4, 3)])
def test_angles(gpu, kind, general):
    rng = np.random.default_rng(4)
    words = np.concatenate([np.arange(1 << 20, dtype=np.uint32), rng.integers(0, 1 << 32, 1 << 22, dtype=np.uint32),
                            (np.arange(1 << 16, dtype=np.uint64) << np.uint64(16)).astype(np.uint32),
                            np.uint32(0xFFFFFFFF) - np.arange(1 << 10, dtype=np.uint32)])
    x = np.float32(6.283185307179586) * (words.astype(np.float32) * np.float32(2.0 ** -32))
    _same_floats(_run(gpu, kind, words), _math(gpu, general, x))


def test_transform_against_the_oracle(gpu):
    import orc
    rng = np.random.default_rng(5)
    n = 1 << 17
    words = np.empty((n, 3), np.uint32)
    words[:, :2] = rng.integers(0, 1 << 32, (n, 2), dtype=np.uint32)
    alpha = np.where(rng.random(n) < 0.5, rng.uniform(0.0, 1.0, n), np.exp(rng.uniform(np.log(1e-6), 0.0, n))).astype(np.float32)
    edge = [0, 1, 0x7FFFFFFF, 0x80000000, 0xFFFFFF00, 0xFFFFFFFF]
    alphas = [1.0, 0.99999994, 1.0 / 255.0, 1e-6, 1e-30, 1e-38]
    k = 0
    for a in alphas:
        for u in edge:
            for v in edge:
                words[k, 0], words[k, 1], alpha[k] = u, v, a
                k += 1
    words[:, 2] = alpha.view(np.uint32)
    u = words[:, :2].astype(np.float32) * np.float32(2.0 ** -32)
    want = np.empty((n, 2), np.float32)
    out = (C.c_float * 2)()
    for i in range(n):
        orc.lib.orc_corrected_box_muller(u[i, 0], u[i, 1], alpha[i], out)
        want[i] = out[0], out[1]
    for kind in (5, 6):
        _same_floats(_run(gpu, kind, words.reshape(-1), n), want[:, kind - 5])
