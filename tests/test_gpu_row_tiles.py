"""The row-tile GEMM (8 rows and more) against the CPU oracle: every tile height, K with and without
splits, ragged rows, columns and groups, each packet format, group size and activation type; captured
calls; activations near the ends of bf16."""

from __future__ import annotations

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.benchmarking.inputs import bf16_bits_to_f32, f16_bits_to_f32, make_case
from fast_kernels.ops import (
    arc_w4a16_forward_native,
    arc_w4a16_plan,
    convert_arc_to_native_packets,
    pack_arc_w4a16_packets,
)
from oracle import oracle

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
FORMATS = {"arc": 0, "native_sym": 1, "native_asym": 2}


def _tensor(bits: np.ndarray, dtype) -> torch.Tensor:
    return torch.from_numpy(bits.view(np.int16).copy()).cuda().view(dtype)


def _packets(case, fmt: str) -> torch.Tensor:
    arc = pack_arc_w4a16_packets(
        torch.from_numpy(case.q_u8).cuda(), _tensor(case.alpha, torch.float16),
        _tensor(case.beta, torch.float16), group_size=case.group_size,
    )
    if fmt == "arc":
        return arc
    return convert_arc_to_native_packets(
        arc, n=case.n, k=case.k, group_size=case.group_size, packet_format=fmt
    )


def _forward(case, x, packets, fmt, output=None):
    return arc_w4a16_forward_native(x, packets, n=case.n, k=case.k, group_size=case.group_size,
                                    packet_format=fmt, output=output)


def _float(y: torch.Tensor) -> np.ndarray:
    return y.float().cpu().numpy().astype(np.float64)


def _check(case, y: torch.Tensor, cols: np.ndarray) -> None:
    """|y - oracle| <= 1e-2 |oracle| + 1e-2 sqrt(K) max alpha, the GEMV bar of the other tests."""
    ref, _ = oracle.gemv(case.x, np.ascontiguousarray(case.q_u8[cols]),
                         np.ascontiguousarray(case.alpha[cols]),
                         np.ascontiguousarray(case.beta[cols]), case.group_size, case.act)
    to_f32 = f16_bits_to_f32 if case.act == "f16" else bf16_bits_to_f32
    ref = to_f32(ref).astype(np.float64)
    bar = 1e-2 * np.abs(ref) + 1e-2 * math.sqrt(case.k) * float(f16_bits_to_f32(case.alpha).max())
    err = np.abs(_float(y)[:, cols] - ref)
    assert np.all(err <= bar), f"max error {err.max():.4g}"


def _check_all(case, y: torch.Tensor) -> None:
    """Every output against the 64-bit product of the dequantised weight: half an ulp of the output, and
    the fp32 sums' own error. Those sums run over (64 or 128 + q) x, at most 143 |x| alpha_max a term, and
    round once per 16 terms within a group and once per group, each by 2^-24 of a partial sum that is
    at most the row's 143 alpha_max sum |x|; 16 of them at full size cover what random signs leave."""
    codes = torch.from_numpy(case.q_u8).cuda()
    codes = torch.stack((codes & 15, codes >> 4), dim=-1).view(case.n, -1, case.group_size)
    alpha, beta = (_tensor(t, torch.float16).double() for t in (case.alpha, case.beta))
    x = _tensor(case.x, DTYPES[case.act]).double()
    want = x @ (codes.double() * alpha[..., None] + beta[..., None]).view(case.n, case.k).t()
    ulp = 2.0**-11 if case.act == "f16" else 2.0**-8
    sums = 16 * 2.0**-24 * 143 * alpha.max() * x.abs().sum(dim=1, keepdim=True)
    err = (y.double() - want).abs()
    assert torch.all(err <= ulp * want.abs() * (1 + 2.0**-6) + sums), f"max error {err.max():.4g}"


# rows, columns, groups by group size, then (m_tile, K split): edges of the tiles (32, 64, 128 rows; 128
# and 256 columns; units of 8 or 16 groups) and one group, among shapes the 16-row tiles are slower
# at; more rows than one launch takes
SHAPES = {
    64: [(17, 16512, 33, (32, False)), (32, 2176, 129, (32, True)), (64, 8320, 40, (64, True)),
         (129, 2176, 129, (64, True)), (300, 6272, 21, (64, False)), (300, 16512, 1, (128, False)),
         (512, 6272, 21, (128, True)), (1025, 3200, 40, (128, True))],
    128: [(9, 128, 21, (32, True)), (16, 2432, 33, (32, True)), (17, 16512, 9, (32, False)), (24, 640, 40, (32, True)), (32, 128, 17, (32, True)),
          (33, 6272, 33, (64, True)), (64, 16512, 8, (64, False)), (96, 3200, 33, (64, True)),
          (300, 6272, 9, (64, False)), (200, 16512, 1, (128, False)), (512, 4224, 17, (128, True)),
          (1025, 640, 65, (64, True))],
}


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("rows,n,groups,group_size,want",
                         [(*s[:3], g, s[3]) for g, shapes in SHAPES.items() for s in shapes])
def test_row_tiles_match_oracle(rows, n, groups, group_size, want, act, fmt) -> None:
    case = make_case(rows, n, groups * group_size, group_size, act=act,
                     asymmetric=fmt != "native_sym", seed=rows + n + groups)
    plan = arc_w4a16_plan(batch=rows, n=n, k=case.k, group_size=group_size,
                          activation_dtype=DTYPES[act], packet_format=FORMATS[fmt])
    assert plan["schedule"] == (4 if rows <= 32 else 3), plan
    on_256_cus = arc_w4a16_plan(batch=rows, n=n, k=case.k, group_size=group_size, cu_count=256,
                                activation_dtype=DTYPES[act], packet_format=FORMATS[fmt])
    assert (on_256_cus["m_tile"], on_256_cus["max_tile_contributors"] > 1) == want
    x = _tensor(case.x, DTYPES[act])
    packets = _packets(case, fmt)
    y = _forward(case, x, packets, fmt)
    # outputs at an odd element offset: no wide stores
    odd = torch.empty(rows * n + 1, device="cuda", dtype=DTYPES[act])[1:].view(rows, n)
    _forward(case, x, packets, fmt, output=odd)
    torch.cuda.synchronize()
    assert torch.equal(y, odd)
    _check(case, y, np.unique(np.linspace(0, n - 1, min(n, 96)).astype(int)))
    _check_all(case, y)


def test_row_tiles_on_two_streams_at_once() -> None:
    """Calls with K splits on two streams whose launches overlap: neither shares counters or partial
    tiles with the other (both schedules)."""
    runs = []
    for rows, n, groups in ((20, 4096, 112), (96, 3200, 33)):
        case = make_case(rows, n, groups * 128, 128, act="bf16", seed=rows)
        x, packets = _tensor(case.x, torch.bfloat16), _packets(case, "native_sym")
        runs.append((case, x, packets, _forward(case, x, packets, "native_sym")))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(3):
        outs = [[], []]
        for _ in range(10):
            for i, stream in enumerate(streams):
                with torch.cuda.stream(stream):
                    for case, x, packets, _ in runs[:: 1 if i else -1]:
                        outs[i].append((case.batch, _forward(case, x, packets, "native_sym")))
        torch.cuda.synchronize()
        want = {case.batch: y for case, _, _, y in runs}
        assert all(torch.equal(y, want[m]) for got in outs for m, y in got)


@pytest.mark.parametrize("rows,n,groups", [(20, 256, 64), (96, 3200, 33)])
def test_row_tiles_in_a_graph(rows, n, groups) -> None:
    """A captured call (K split, so with counters and partial tiles) replays to the eager bits, with
    eager work in between."""
    case = make_case(rows, n, groups * 128, 128, act="bf16", seed=7)
    assert arc_w4a16_plan(batch=rows, n=n, k=case.k, group_size=128, activation_dtype=torch.bfloat16,
                          packet_format=1)["schedule"] == (4 if rows <= 32 else 3)
    x = _tensor(case.x, torch.bfloat16)
    packets = _packets(case, "native_sym")
    want = _forward(case, x, packets, "native_sym")
    out = torch.zeros_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _forward(case, x, packets, "native_sym", output=out)
    for _ in range(4):
        out.zero_()
        graph.replay()
        again = _forward(case, x, packets, "native_sym")
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(again, want)


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("exponent", [-100, 100, 120])
@pytest.mark.parametrize("rows,n,groups", [(18, 256, 64), (96, 3200, 33)])
def test_row_tiles_at_the_ends_of_bf16(rows, n, groups, exponent, fmt) -> None:
    """Activations scaled by 2^exponent scale the outputs: to 2^120, where sums of (128 + q) x pass
    the largest fp32, and a row with an infinity is not finite while the others are untouched."""
    case = make_case(rows, n, groups * 128, 128, act="bf16", asymmetric=fmt != "native_sym", seed=5)
    x = _tensor(case.x, torch.bfloat16)
    packets = _packets(case, fmt)
    want = _forward(case, x, packets, fmt)
    scaled = (x.double() * 2.0**exponent).to(torch.bfloat16)
    got = _forward(case, scaled, packets, fmt)
    assert torch.isfinite(got).all()
    err = (got.double() * 2.0**-exponent - want.double()).abs()
    # two roundings to bf16 of sums that may be taken in another order
    bar = want.double().abs() * 2.0**-7 + 1e-3 * want.double().square().mean().sqrt()
    assert torch.all(err <= bar)
    scaled[3, 17] = math.inf
    again = _forward(case, scaled, packets, fmt)
    assert not torch.isfinite(again[3]).any()
    keep = [r for r in range(rows) if r != 3]
    assert torch.equal(again[keep], got[keep])


@pytest.mark.parametrize("rows", [32, 64, 512])
@pytest.mark.parametrize("value", [math.nan, math.inf])
def test_a_non_finite_row_costs_little(rows, value) -> None:
    """A row that holds a NaN (a padded one, say) leaves a bf16 call's time as it is: nothing is
    computed again for it. At most three times, for the clock's sake; again by one lane an output it
    would be fifty times and more."""
    n, k = 28672, 4096
    case = make_case(1, 128, k, 128, act="bf16", seed=1)
    x = torch.randn((rows, k), device="cuda").to(torch.bfloat16)
    packets = _packets(case, "native_sym").repeat(n // 128, 1)
    case.n = n
    bad = x.clone()
    bad[rows // 2, 5] = value
    times = []
    for inputs in (x, bad, x, bad):
        _forward(case, inputs, packets, "native_sym")
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(10):
            out = _forward(case, inputs, packets, "native_sym")
        end.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(end) * 100.0)
    print("us a call:", [round(t, 1) for t in times])
    assert min(times[1], times[3]) <= 3 * min(times[0], times[2])
    assert not torch.isfinite(out[rows // 2]).any()
    rest = [r for r in range(rows) if r != rows // 2]
    assert torch.equal(out[rest], _forward(case, x, packets, "native_sym")[rest])
