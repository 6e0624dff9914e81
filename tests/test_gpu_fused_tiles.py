"""The fused decode-step neighbours on the row tiles against a dense product that shares no code with
them: torch's RMSNorm, the dequantised weight in 64 bits, torch's SiLU. Every tile height with SiLU's
gate and up columns, K with and without splits, ragged rows, more rows than one launch takes; and the
calls a workspace that is too small for them."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.native import native_module
from fast_kernels.ops import (
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
    zp = torch.full((n, k // g), 8, device="cuda", dtype=torch.uint8)
    if fmt == "native_asym":
        zp = torch.randint(0, 16, (n, k // g), generator=gen, device="cuda", dtype=torch.uint8)
    slabs = pack_native_w4a16_packets(q, alpha, zp if fmt == "native_asym" else None, group_size=g,
                                      packet_format=fmt)
    codes = torch.stack((q & 15, q >> 4), dim=-1).view(n, k // g, g)
    beta = (-(alpha.float() * zp.float())).half()
    dense = (codes.double() * alpha.double()[..., None] + beta.double()[..., None]).view(n, k)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dtype)
    gamma = (torch.rand(k, generator=gen, device="cuda") + 0.5).to(dtype)
    return x, gamma, slabs, dense, dict(n=n, k=k, group_size=g, packet_format=fmt)


def _norm(x, gamma):
    h = (x.float() * torch.rsqrt(x.float().square().mean(-1, keepdim=True) + EPS)).to(x.dtype)
    return (gamma.float() * h.float()).to(x.dtype)


def _assert_close(got, want, bits):
    """Norm, product and SiLU are rounded to the activation type on both sides; fp32 sums against 64-bit
    ones flip some of those roundings. A flipped one is 2^-bits of its value, and three of them meet
    in an output; the norm's travel through a product of K terms and stay far below its rms."""
    want = want.float()
    rms = want.square().mean().sqrt()
    err = (got.float() - want).abs()
    assert torch.all(err <= 4 * 2.0**-bits * (want.abs() + rms)), f"max {err.max():.4g} rms {rms:.4g}"


# rows, n, K groups, group size, then (tile height, K split) with SiLU on 256 CUs
CASES = [
    (129, 16384, 5, 64, (128, False)), (300, 8192, 33, 64, (128, True)),
    (300, 8192, 5, 128, (128, False)), (200, 16384, 8, 128, (128, False)),
    (512, 8192, 17, 128, (128, True)), (1030, 2304, 17, 128, (128, True)),
    (1100, 4096, 17, 64, (128, True)), (20, 8192, 17, 128, None), (70, 4096, 33, 64, None),
]


@pytest.mark.parametrize("fmt", ["native_sym", "native_asym"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,groups,g,want", CASES)
def test_fused_row_tiles_match_a_dense_product(rows, n, groups, g, want, dtype, fmt) -> None:
    bits = 10 if dtype == torch.float16 else 7
    code, act = (2 if fmt == "native_asym" else 1), int(dtype == torch.bfloat16)
    for silu in (False, True):
        plan = native_module().w4a16_plan_fused(rows, n, groups * g, g, act, 256, code, silu)
        assert plan["schedule"] == 3, plan
        if want:
            # a plan of more rows than one launch takes is that of its full launches
            assert (plan["m_tile"], plan["max_tile_contributors"] > 1) == want, plan
    x, gamma, slabs, dense, shape = _case(rows, n, groups * g, g, dtype, fmt)
    xn = _norm(x, gamma)
    y = (xn.double() @ dense.t()).to(dtype)
    _assert_close(arc_w4a16_forward_rmsnorm(x, gamma, slabs, eps=EPS, **shape), y, bits)
    gate, up = y[:, : n // 2].float(), y[:, n // 2 :].float()
    act_mul = (torch.nn.functional.silu(gate).to(dtype).float() * up).to(dtype)
    _assert_close(arc_w4a16_forward_silu_mul(x, slabs, norm_weight=gamma, eps=EPS, **shape),
                  act_mul, bits)
    _assert_close(arc_w4a16_forward_silu_mul(xn, slabs, **shape), act_mul, bits)


def test_a_workspace_too_small_is_refused() -> None:
    """Both row-tile schedules and a fused call, one byte short: ValueError before any launch."""
    native = native_module()
    n, k, g = 4096, 14336, 128
    ws = torch.zeros(64 << 20, device="cuda", dtype=torch.uint8)
    x, gamma, slabs, _, _ = _case(64, n, k, g, torch.float16, "native_sym")
    out = torch.zeros((64, n), device="cuda", dtype=torch.float16)
    for rows, schedule in ((20, 4), (64, 3)):
        plan = native.arc_w4a16_plan(rows, n, k, g, 0, 0, 0, 1, 0)
        assert plan["schedule"] == schedule and 0 < plan["workspace_bytes"] <= ws.numel()
        for short, refused in ((1, True), (0, False)):
            args = (x.data_ptr(), slabs.data_ptr(), out.data_ptr(), ws.data_ptr(),
                    plan["workspace_bytes"] - short, rows, n, k, g, 1, 0, 0, 0)
            if refused:
                with pytest.raises(ValueError, match="workspace_bytes"):
                    native.arc_w4a16_forward_native(*args)
            else:
                native.arc_w4a16_forward_native(*args)
    plan = native.w4a16_plan_fused(64, n, k, g, 0, 0, 1, True)
    assert plan["schedule"] == 3
    with pytest.raises(ValueError, match="workspace_bytes"):
        native.w4a16_forward_fused(x.data_ptr(), gamma.data_ptr(), EPS, slabs.data_ptr(),
                                   out.data_ptr(), ws.data_ptr(), plan["workspace_bytes"] - 1, 64, n,
                                   k, g, 1, 0, True, 0)
    torch.cuda.synchronize()
