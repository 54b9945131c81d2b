"""Host rules that size launches (no GPU): rows per unit of the two-column
streaming kernel, rows per thread of the single-pass tile kernel."""
import numpy as np
import pytest

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
