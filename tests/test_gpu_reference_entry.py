"""The reference-signature forward (no workspace argument, library-owned memory) at rows that the
row tiles take: captured calls, and calls on several streams."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.native import native_module
from fast_kernels.ops import arc_packet_stride_bytes, arc_w4a16_forward, pack_arc_w4a16_packets

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

G = 128


def _case(rows, n, k, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed + rows + n + k)
    q = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    alpha = (torch.rand((n, k // G), generator=gen, device="cuda") * 0.019 + 0.001).half()
    beta = (-8.0 * alpha.float()).half()
    x = torch.randn((rows, k), generator=gen, device="cuda").half()
    return x, pack_arc_w4a16_packets(q, alpha, beta, group_size=G)


def _call(x, packets, out, stream) -> None:
    native_module().arc_w4a16_forward(x.data_ptr(), packets.data_ptr(), 0, out.data_ptr(),
                                      x.shape[0], out.shape[1], x.shape[1], G,
                                      arc_packet_stride_bytes(G), stream.cuda_stream)


def _new_out(x, n):
    return torch.zeros((x.shape[0], n), device="cuda", dtype=torch.float16)


def test_captured_call_of_a_plan_without_workspace() -> None:
    """16 rows x 22016 x 4096: the row tiles need no memory there, the 16-row tiles do; after a
    warm-up the call captures and replays to the eager bits."""
    rows, n, k = 16, 22016, 4096
    x, packets = _case(rows, n, k)
    stream = torch.cuda.Stream()
    want, out = _new_out(x, n), _new_out(x, n)
    torch.cuda.synchronize()
    _call(x, packets, want, stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _call(x, packets, out, stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
