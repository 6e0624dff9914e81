"""Which kernel a plan takes at measured shapes (256 CUs): the row tiles only where they are the faster
ones. Schedules: 0 the 16-row tiles or the dot2 runs, 3 and 4 the row tiles."""

from __future__ import annotations

import pytest

from fast_kernels.native import native_module


def _schedule(rows, n, k, g, fmt) -> int:
    return native_module().arc_w4a16_plan(rows, n, k, g, 0, 0, 256, fmt, 0)["schedule"]


@pytest.mark.parametrize("rows,n,k,g,fmt", [(39, 11520, 1920, 128, 2), (72, 6656, 1920, 128, 0)])
def test_workgroups_just_past_a_round_stay_on_16_row_tiles(rows, n, k, g, fmt) -> None:
    """14.9 us against 17.9 on the row tiles, and 14.3 against 16.8."""
    assert _schedule(rows, n, k, g, fmt) == 0


@pytest.mark.parametrize("rows,n,k,g,fmt,want", [
    (33, 22016, 4096, 128, 0, 3), (64, 4096, 14336, 128, 1, 3), (512, 10240, 8192, 128, 1, 3),
    (48, 3200, 16064, 64, 0, 3), (46, 13696, 3200, 128, 0, 3), (20, 4096, 14336, 128, 1, 4),
    (17, 16512, 2112, 64, 0, 4), (64, 8320, 2560, 64, 1, 3),
])
def test_row_tiles_keep_what_they_are_faster_at(rows, n, k, g, fmt, want) -> None:
    assert _schedule(rows, n, k, g, fmt) == want
