"""Packing and dequantising kernels against plain tensor indexing, byte for byte: K of whole and part
turns (256 values a workgroup pass), one to several passes a workgroup, odd group counts."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.ops import (
    convert_arc_to_native_packets,
    convert_native_to_arc_packets,
    dequant_arc_w4a16_packets_to_fp16,
    pack_arc_w4a16_packets,
    pack_native_w4a16_packets,
)

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _reference_packets(q, alpha, beta, g):
    """[(N/128) * K/G, 64 G + 512]: word w of column c at byte (w * 128 + c) * 4, alphas, betas."""
    n, groups = alpha.shape
    words = q.view(torch.int32).view(n // 128, 128, groups, g // 8)
    codes = words.permute(0, 2, 3, 1).contiguous().view(torch.uint8).view(n // 128, groups, -1)
    scales = [t.view(n // 128, 128, groups).transpose(1, 2).contiguous().view(torch.uint8)
              .view(n // 128, groups, -1) for t in (alpha, beta)]
    return torch.cat([codes, *scales], dim=2).view(n // 128 * groups, -1)


@pytest.mark.parametrize("n,groups,g", [(128, 1, 64), (128, 1, 128), (256, 3, 128), (384, 7, 64),
                                        (1024, 33, 128), (4096, 64, 64), (33792, 8, 128),
                                        (16384, 43, 64)])
def test_packets_byte_for_byte(n, groups, g) -> None:
    gen = torch.Generator(device="cuda").manual_seed(n + groups)
    k = groups * g
    q = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    # from 0.001 up: with alpha = 0 every zero point gives the same beta, and the conversion back to
    # zero points (the smallest that fits) is not the one packed
    alpha = (torch.rand((n, groups), generator=gen, device="cuda") * 0.019 + 0.001).half()
    zp = torch.randint(0, 16, (n, groups), generator=gen, device="cuda", dtype=torch.uint8)
    beta = (-(alpha.float() * zp.float())).half()
    shape = dict(n=n, k=k, group_size=g)
    arc = pack_arc_w4a16_packets(q, alpha, beta, group_size=g)
    assert torch.equal(arc, _reference_packets(q, alpha, beta, g))

    codes = torch.stack((q & 15, q >> 4), dim=-1).view(n, groups, g)
    dense = (codes.double() * alpha.double()[..., None] + beta.double()[..., None]).half().view(n, k)
    assert torch.equal(dequant_arc_w4a16_packets_to_fp16(arc, **shape), dense)

    native = pack_native_w4a16_packets(q, alpha, zp, group_size=g, packet_format="native_asym")
    assert torch.equal(native, convert_arc_to_native_packets(arc, packet_format="native_asym", **shape))
    assert torch.equal(convert_native_to_arc_packets(native, packet_format="native_asym", **shape), arc)
    sym = pack_native_w4a16_packets(q, alpha, group_size=g, packet_format="native_sym")
    eight = (-8.0 * alpha.float()).half()
    assert torch.equal(convert_native_to_arc_packets(sym, packet_format="native_sym", **shape),
                       pack_arc_w4a16_packets(q, alpha, eight, group_size=g))
