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


def _fused(rows, n, k, g, silu) -> int:
    return native_module().w4a16_plan_fused(rows, n, k, g, 0, 256, 1, silu)["schedule"]


@pytest.mark.parametrize("rows,n,k,g,silu", [
    (4, 34816, 1408, 64, True), (3, 43776, 1472, 64, True), (5, 7296, 1280, 128, False),
    (9, 3584, 1280, 128, False), (7, 4736, 1856, 64, False), (5, 4096, 1024, 128, False),
])
def test_fused_calls_of_short_k_stay_on_dot2_kernels(rows, n, k, g, silu) -> None:
    """In us, dot2 and row tiles: 15.8 and 31.5, 21.7 and 32.8, 9.5 and 13.4, 9.7 and 13.0, 12.4 and
    15.7, 8.3 and 10.9."""
    assert _fused(rows, n, k, g, silu) == 0


@pytest.mark.parametrize("rows,n,k,g,silu", [
    (13, 32640, 3328, 128, False), (11, 2304, 20160, 64, False), (8, 5760, 2560, 128, False),
    (5, 1152, 4032, 64, False), (3, 32000, 1664, 128, True), (15, 3584, 1664, 128, True),
])
def test_fused_calls_keep_the_row_tiles_where_faster(rows, n, k, g, silu) -> None:
    assert _fused(rows, n, k, g, silu) == 3


@pytest.mark.parametrize("act,n,k,want", [
    (1, 2048, 2048, 0), (1, 8192, 2048, 0), (0, 8192, 2048, 2), (1, 24576, 2048, 2), (1, 2048, 4096, 2),
])
def test_two_bf16_rows_of_short_k_stay_on_dot2(act, n, k, want) -> None:
    """RMSNorm at 2 rows, dot2 and matrix cores in us: 5.5 and 6.0, 5.8 and 6.5; fp16 5.5 and 5.4; one
    and a half slices per CU 11.3 and 9.2."""
    plan = native_module().w4a16_plan_fused(2, n, k, 128, act, 256, 1, False)
    assert plan["schedule"] == want
