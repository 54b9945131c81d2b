"""Host rules that size launches (no GPU): rows per unit of the two-column
streaming kernel, rows per thread of the single-pass tile kernel."""
import numpy as np
import pytest
import torch

from opymize_amd.solvers import autotune, tv


@pytest.mark.parametrize("k", [2, 4, 8])
@pytest.mark.parametrize("shapes", [[(1, 1)], [(64, 64)], [(256, 256)], [(512, 512)], [(1024, 1024)], [(3, 5000)],
                                    [(5000, 3)], [(100, 100)] * 16, [(64, 64)] * 300, [(1024, 1024)] * 32])
def test_wide_rows_fill_the_chip(shapes, k):
    """No more rows per unit than leave half the SIMDs with one, down to one row."""
    H, W = np.array([s[0] for s in shapes]), np.array([s[1] for s in shapes])
    strips = tv._wide_strips(W, tv.WIDE_COLS - 2 * k)
    rows = tv.wide_rows(H, strips, k, 1024)
    units = int(np.sum(strips * -(-H // rows)))
    if np.sum(strips * H) <= 1024:
        assert rows == 1
    else:
        assert units >= 512


def test_wide_rows_pass_over_empty_images():
    H, W = np.array([0, 700, 300, 0]), np.array([5, 900, 400, 0])
    strips = tv._wide_strips(W, 112)
    assert tv.wide_rows(H, strips, 8, 1024) == tv.wide_rows(H[1:3], strips[1:3], 8, 1024)


@pytest.mark.parametrize("n,H,W,k", [(4, 1024, 1024, 8), (4, 1024, 1024, 6), (1, 2048, 2048, 6), (2, 2048, 2048, 6),
                                     (12, 1024, 1024, 8)])
def test_wide_rows_leave_no_handful_over(n, H, W, k):
    """A few units beside two full ones per SIMD start when the others end and
    take as long again: not one to a hundredth of the SIMDs over."""
    h, w = np.full(n, H), np.full(n, W)
    strips = tv._wide_strips(w, tv.WIDE_COLS - 2 * k)
    units = int(np.sum(strips * -(-h // tv.wide_rows(h, strips, k, 1024))))
    assert not 2048 < units < 2048 + 11


def test_kernel_choice_does_not_walk_the_batch():
    """The choice is made several times per block: its cost must not grow with
    the number of instances."""
    class Shapes(list):
        closed = False

        def __iter__(self):
            assert not self.closed, "walked the instances"
            return list.__iter__(self)

    bat = object.__new__(tv.TVBatch)
    bat.C, bat.dtype, bat.multi, bat.multi_kernel, bat._wide_now, bat._stream_now = 1, torch.float32, 8, "auto", True, True
    cfg = tv.TVCfg()
    cfg.steps = tv.STEP_MODES["accel"]
    shapes = Shapes([(64, 64), (30, 500)])
    bat.shapes = shapes
    bat._shapes, shapes.closed = shapes, True
    assert bat._use_wide(cfg) and bat._use_stream(cfg) and bat._launch_k(cfg) == 8
    bat.shapes = [(64, 64), (23171, 23171)]  # 2 x 4 B x 23171^2 > 2^32
    assert not bat._use_wide(cfg)


@pytest.mark.parametrize("C", [1, 2, 3, 4])
@pytest.mark.parametrize("H,W", [(1, 1), (64, 64), (128, 128), (256, 256), (512, 512), (1024, 1024), (2048, 2048),
                                 (7, 9000), (9000, 7)])
def test_default_tile_rows(H, W, C):
    """The full rows per thread where they give a tile per CU, else the most
    that do, down to one; the tile heights the kernels are built for."""
    tw, rpt = autotune.default_tile(H, W, C)
    full = 8 if C == 1 else 4
    tiles = lambda r: -(-H // (4 * r)) * -(-W // 64)  # noqa: E731
    assert tw == 64 and rpt in (1, 2, 4, 8) and rpt <= full
    assert rpt == 1 or tiles(rpt) >= 256
    assert rpt == full or tiles(2 * rpt) < 256
