"""The distributor's tile sums at the edges of a tile and on both sides of the
number of tiles that take a scan launch, over frames that reuse the sums."""
import numpy as np
import pytest

import helpers as H
from helpers import assert_same, flush

pytestmark = pytest.mark.gpu

TILE = 4096
FOLD = 1024  # tiles up to which the distribute workgroups add the sums up themselves


def _frames(gpu, w, h, **kw):
    # the second frame looks away: a pass without points
    eyes = [((0.0, 1.0, -12.0), (0, 0, 0)), ((0.0, 1.0, -12.0), (0, 0, -99)), ((2.0, 1.0, -11.0), (0, 0, 0))]
    return [gpu.frame_params(e, t, (0, 1, 0), 45.0, w, h, ss=1, frame=i, **kw) for i, (e, t) in enumerate(eyes)]


@pytest.mark.parametrize("budget", [10_000_000, 3_000])
@pytest.mark.parametrize("n", [1, TILE - 1, TILE, TILE + 1, 257 * TILE + 3])
def test_tiles_against_the_oracle(gpu, n, budget):
    arrays = H.scene(0x5EED0901, n, dict(H.C1, half_extent=3.0, log_scale_mu=-3.5))
    st = gpu.RenderSettings(160, 90, 1, 1, max_number_of_points=budget)
    a, b = H.GpuRunner(arrays, st), H.OracleRunner(arrays, st)
    for i, f in enumerate(_frames(gpu, 160, 90, occlusion=True)):
        flush(f"tiles n {n} budget {budget} frame {i}")
        x, y = a.render(f, H.INTERMEDIATES), b.render(f, H.INTERMEDIATES)
        assert x.stats["num_points"] == y.stats["num_points"], (x.stats, y.stats)
        for k in H.INTERMEDIATES:
            assert_same(f"n {n} frame {i} {k}", x.debug[k], y.debug[k])
        assert_same(f"n {n} frame {i} colour", x.color, y.color)


def test_both_sides_of_the_scan_launch(gpu):
    n = FOLD * TILE
    arrays = H.scene(0x5EED0911, n + 1, dict(H.C1, half_extent=8.0, log_scale_mu=-5.0))
    arrays.means[n] = (0.0, 500.0, 0.0)  # in no view
    arrays.scales[n] = 0.01
    st = gpu.RenderSettings(640, 360, 1, 1)
    with_scan, folded = H.GpuRunner(arrays, st), H.GpuRunner(arrays.subset(np.arange(n)), st)
    for i, f in enumerate(_frames(gpu, 640, 360)):
        flush(f"tiles n {n} frame {i}")
        which = [gpu.DBG_VALID_IDS, gpu.DBG_VALID_OFFSETS, gpu.DBG_FRAMEBUFFER]
        x, y = folded.render(f, which), with_scan.render(f, which)
        assert x.stats["num_points"] == y.stats["num_points"] and (i == 1) == (x.stats["num_points"][0] == 0)
        for k in which:
            assert_same(f"frame {i} {k}", x.debug[k], y.debug[k])
