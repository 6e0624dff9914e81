"""Captured calls of the Python ops that need a zero-filled workspace (K splits): each graph has its
own, whatever eager calls on the stream and other graphs do."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from conftest import gpu_available
from fast_kernels.ops import (
    arc_w4a16_forward,
    arc_w4a16_forward_native,
    arc_w4a16_plan,
    convert_arc_to_native_packets,
    pack_arc_w4a16_packets,
)

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

G = 128


def _case(rows, n, k):
    gen = torch.Generator(device="cuda").manual_seed(rows + n + k)
    q = torch.randint(0, 256, (n, k // 2), generator=gen, device="cuda", dtype=torch.uint8)
    alpha = (torch.rand((n, k // G), generator=gen, device="cuda") * 0.019 + 0.001).half()
    arc = pack_arc_w4a16_packets(q, alpha, (-8.0 * alpha.float()).half(), group_size=G)
    x = torch.randn((rows, k), generator=gen, device="cuda").half()
    return x, arc, convert_arc_to_native_packets(arc, n=n, k=k, group_size=G)


def _needs(rows, n, k, packet_format) -> int:
    return arc_w4a16_plan(batch=rows, n=n, k=k, group_size=G, packet_format=packet_format)["workspace_bytes"]


def _graph(call, out, stream):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(out)
    return graph


# rows, n, k, format: 16-row tiles and direct row tiles with K splits
SMALL = [(9, 256, 8192, 0), (20, 256, 8192, 1), (20, 4096, 14336, 1)]


@pytest.mark.parametrize("rows,n,k,fmt", SMALL)
def test_graphs_keep_their_own_workspace(rows, n, k, fmt) -> None:
    x, arc, native = _case(rows, n, k)
    big_x, _, big_native = _case(32, 8192, 28672)
    assert 0 < _needs(rows, n, k, fmt) < _needs(32, 8192, 28672, 1)

    def call(out):
        if fmt == 0:
            arc_w4a16_forward(x, arc, n=n, k=k, group_size=G, output=out)
        else:
            arc_w4a16_forward_native(x, native, n=n, k=k, group_size=G, output=out)

    stream = torch.cuda.Stream()
    want, first, second = (torch.zeros((rows, n), device="cuda", dtype=torch.float16) for _ in range(3))
    call(want)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call(want)  # the stream's eager workspace
    torch.cuda.synchronize()
    graphs = [_graph(call, first, stream), _graph(call, second, stream)]
    outs = [first, second]
    for turn in (1, 0, 1, 0):  # the graph captured last replays first
        with torch.cuda.stream(stream):
            big = arc_w4a16_forward_native(big_x, big_native, n=8192, k=28672, group_size=G)
            others = [torch.full((1 << 20,), 7, device="cuda", dtype=torch.uint8) for _ in range(8)]
            outs[turn].zero_()
            graphs[turn].replay()
            again = arc_w4a16_forward_native(big_x, big_native, n=8192, k=28672, group_size=G)
        torch.cuda.synchronize()
        assert torch.equal(outs[turn], want) and torch.equal(big, again)
        assert all(bool((t == 7).all()) for t in others)


def test_calls_of_one_graph_share_a_workspace() -> None:
    x, _, native = _case(20, 4096, 14336)
    want = arc_w4a16_forward_native(x, native, n=4096, k=14336, group_size=G)
    outs = [torch.zeros_like(want) for _ in range(3)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    before = torch.cuda.memory_allocated()
    with torch.cuda.graph(graph):
        for out in outs:
            arc_w4a16_forward_native(x, native, n=4096, k=14336, group_size=G, output=out)
    held = torch.cuda.memory_allocated() - before
    assert held <= 2 * _needs(20, 4096, 14336, 1)
    for _ in range(3):
        for out in outs:
            out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(out, want) for out in outs)
