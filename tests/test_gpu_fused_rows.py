"""The fused decode-step neighbours at several rows (the matrix-core stream kernel and the row-tile
GEMM) against the unfused pipeline: torch's RMSNorm, the plain forward, torch's SiLU and product."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.native import native_module
from fast_kernels.ops import (
    arc_w4a16_forward_native,
    arc_w4a16_forward_rmsnorm,
    arc_w4a16_forward_silu_mul,
    pack_native_w4a16_packets,
)

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

EPS = 1e-5


def _case(rows, n, k, g, dtype, fmt):
    gen = torch.Generator(device="cuda").manual_seed(rows * 1000 + n + k)
    q = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    alpha = (torch.rand((n, k // g), generator=gen, device="cuda") * 0.019 + 0.001).half()
    zp = None
    if fmt == "native_asym":
        zp = torch.randint(0, 16, (n, k // g), generator=gen, device="cuda", dtype=torch.uint8)
    slabs = pack_native_w4a16_packets(q, alpha, zp, group_size=g, packet_format=fmt)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dtype)
    gamma = (torch.rand(k, generator=gen, device="cuda") + 0.5).to(dtype)
    return x, gamma, slabs, dict(n=n, k=k, group_size=g, packet_format=fmt)


def _norm(x, gamma):
    h = (x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + EPS)).to(x.dtype)
    return (gamma.float() * h.float()).to(x.dtype)


def _assert_close(got, want, bits):
    """Both sides round the norm, the product (and the SiLU) to the activation type; sums in another
    order flip some of those roundings. A flipped one is 2^-bits of its value, and three of them meet
    in an output; the norm's travel through a product of K terms and stay far below its rms."""
    want = want.float()
    rms = want.square().mean().sqrt()
    err = (got.float() - want).abs()
    assert torch.all(err <= 4 * 2.0**-bits * (want.abs() + rms)), f"max {err.max():.4g} rms {rms:.4g}"


# rows, n, k in groups, then (m_tile, schedule) on 256 CUs: the stream kernel at its row steps (4, 8,
# 16) and unit counts (fewer than the CUs, one each, several), and the row tiles where K is long or
# ragged, the slices do not divide, or the rows are many
CASES = [
    (2, 2048, 32, 128, (16, 2)), (4, 6144, 32, 128, (16, 2)), (5, 1024, 16, 128, (16, 2)),
    (8, 28672, 32, 128, (16, 2)), (9, 14336, 32, 64, (16, 2)), (16, 16384, 32, 128, (16, 2)),
    (3, 8192, 86, 128, (32, 3)), (6, 4096, 21, 128, (32, 3)), (16, 11008, 43, 64, (32, 3)),
    (17, 512, 33, 128, (32, 3)), (40, 2304, 65, 64, (64, 3)), (130, 1024, 16, 128, None),
    (40, 512, 8, 128, (8, 0)),
]


@pytest.mark.parametrize("fmt", ["native_sym", "native_asym"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,groups,g,want", CASES)
def test_fused_rows_match_unfused_pipeline(rows, n, groups, g, want, dtype, fmt) -> None:
    bits = 10 if dtype == torch.float16 else 7
    x, gamma, slabs, shape = _case(rows, n, groups * g, g, dtype, fmt)
    xn = _norm(x, gamma)
    y = arc_w4a16_forward_native(xn, slabs, **shape)
    if want and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        code = 2 if fmt == "native_asym" else 1
        plan = native_module().w4a16_plan_fused(rows, n, groups * g, g, 0, 0, code, False)
        assert (plan["m_tile"], plan["schedule"]) == want, plan
    got = arc_w4a16_forward_rmsnorm(x, gamma, slabs, eps=EPS, **shape)
    _assert_close(got, y, bits)
    assert torch.equal(got, arc_w4a16_forward_rmsnorm(x, gamma, slabs, eps=EPS, **shape))
    gate, up = y[:, : n // 2].float(), y[:, n // 2 :].float()
    act = torch.nn.functional.silu(gate).to(dtype).float()
    _assert_close(arc_w4a16_forward_silu_mul(x, slabs, norm_weight=gamma, eps=EPS, **shape),
                  (act * up).to(dtype), bits)
    _assert_close(arc_w4a16_forward_silu_mul(xn, slabs, **shape), (act * up).to(dtype), bits)
