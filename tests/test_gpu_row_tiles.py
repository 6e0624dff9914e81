"""The row-tile GEMM (17 rows and more) against the CPU oracle: every tile height, K with and without
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


# rows, columns, groups: edges of the tiles (32, 64, 128 rows; 128 and 256 columns; units of 8 or
# 16 groups), one group, K split and not, more rows than one launch takes
SHAPES = [(17, 128, 1), (32, 256, 3), (33, 384, 17), (64, 1152, 21), (65, 640, 40), (129, 256, 33),
          (200, 4224, 8), (1025, 128, 5)]


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("group_size", [64, 128])
@pytest.mark.parametrize("act", ["f16", "bf16"])
@pytest.mark.parametrize("rows,n,groups", SHAPES)
def test_row_tiles_match_oracle(rows, n, groups, act, group_size, fmt) -> None:
    case = make_case(rows, n, groups * group_size, group_size, act=act,
                     asymmetric=fmt != "native_sym", seed=rows + n + groups)
    plan = arc_w4a16_plan(batch=rows, n=n, k=case.k, group_size=group_size,
                          activation_dtype=DTYPES[act], packet_format=FORMATS[fmt])
    assert plan["schedule"] == 3, plan
    x = _tensor(case.x, DTYPES[act])
    packets = _packets(case, fmt)
    y = _forward(case, x, packets, fmt)
    # outputs at an odd element offset: no wide stores
    odd = torch.empty(rows * n + 1, device="cuda", dtype=DTYPES[act])[1:].view(rows, n)
    _forward(case, x, packets, fmt, output=odd)
    torch.cuda.synchronize()
    assert torch.equal(y, odd)
    _check(case, y, np.unique(np.linspace(0, n - 1, min(n, 96)).astype(int)))


@pytest.mark.parametrize("rows,n,groups", [(40, 512, 40), (20, 256, 64)])
def test_row_tiles_in_a_graph(rows, n, groups) -> None:
    """A captured call (K split, so with counters and partial tiles) replays to the eager bits, with
    eager work in between."""
    case = make_case(rows, n, groups * 128, 128, act="bf16", seed=7)
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
def test_row_tiles_at_the_ends_of_bf16(exponent, fmt) -> None:
    """Activations scaled by 2^exponent scale the outputs: to 2^120, where sums of (128 + q) x pass
    the largest fp32, and a row with an infinity is not finite while the others are untouched."""
    case = make_case(18, 256, 512, 128, act="bf16", asymmetric=fmt != "native_sym", seed=5)
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
    keep = [r for r in range(18) if r != 3]
    assert torch.equal(again[keep], got[keep])
