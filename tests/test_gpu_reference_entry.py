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


# rows, n, k: row tiles that need prepared activations (no K split and K splits), and ones that need
# only partial tiles; the 16-row tiles need no memory at the first and the fourth
CAPTURED = [(33, 22016, 4096), (96, 3200, 4224), (20, 4096, 14336), (300, 2048, 8192)]


@pytest.mark.parametrize("rows,n,k", CAPTURED)
def test_captured_call_survives_larger_calls(rows, n, k) -> None:
    """A graph of the call replays to the same bits after the stream's memory has grown for calls of
    more rows, and after that memory is given back; the call captured is the one without row tiles."""
    x, packets = _case(rows, n, k)
    more, more_packets = _case(600, 10240, 8192)
    stream = torch.cuda.Stream()
    out, more_out = _new_out(x, n), _new_out(more, 10240)
    torch.cuda.synchronize()
    _call(x, packets, out, stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _call(x, packets, out, stream)
    want = arc_w4a16_forward(x, packets, n=n, k=k, group_size=G, impl="mfma")  # 16-row tiles
    torch.cuda.synchronize()
    more_want = None
    for step in range(4):
        _call(more, more_packets, more_out, stream)
        torch.cuda.synchronize()
        more_want = more_out.clone() if more_want is None else more_want
        assert torch.equal(more_out, more_want)
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        if step == 1:
            native_module().release_workspaces()


def test_row_tiles_on_many_streams_at_once() -> None:
    """More streams than the library keeps memory for, calls of two sizes (a K split whose counters
    and partial tiles must not be shared; more rows than one launch's memory allows) interleaved."""
    runs = []
    for rows, n, k in ((96, 3200, 4224), (20, 4096, 14336), (1100, 1024, 57344)):
        x, packets = _case(rows, n, k)
        runs.append((x, packets, arc_w4a16_forward(x, packets, n=n, k=k, group_size=G)))
    streams = [torch.cuda.Stream() for _ in range(10)]
    torch.cuda.synchronize()
    for _ in range(2):
        outs = []
        for stream in streams:
            for x, packets, want in runs:
                out = torch.zeros_like(want)
                stream.wait_stream(torch.cuda.current_stream())
                _call(x, packets, out, stream)
                outs.append((out, want))
        torch.cuda.synchronize()
        for out, want in outs:
            # both round sums of the same products to fp16 once, in another order
            assert (out.float() - want.float()).abs().max() <= 2.0**-9 * want.float().abs().max()
    native_module().release_workspaces()


def test_eager_call_while_another_stream_captures() -> None:
    """The first call on a stream allocates; a capture under way on another stream goes on."""
    x, packets = _case(96, 3200, 4224)
    want = arc_w4a16_forward(x, packets, n=3200, k=4224, group_size=G)
    stream = torch.cuda.Stream()
    out, a = torch.zeros_like(want), torch.ones(1024, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        b = a + 1
        _call(x, packets, out, stream)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(b, a + 1)


def test_too_many_units_are_refused() -> None:
    """batch * (n / 32) * (k / group_size) from 2^31 on is refused before any launch, by the row tiles
    as by the other kernels."""
    x, packets = _case(17, 57344, 8192)
    out = _new_out(x, 57344)
    rows = 2**31 // (57344 // 32 * (8192 // G)) + 1
    with pytest.raises(ValueError, match="2\\^31"):
        native_module().arc_w4a16_forward(x.data_ptr(), packets.data_ptr(), 0, out.data_ptr(), rows,
                                          57344, 8192, G, arc_packet_stride_bytes(G), 0)
    with pytest.raises(ValueError, match="2\\^31"):
        native_module().w4a16_forward_fused(x.data_ptr(), x.data_ptr(), 1e-5, packets.data_ptr(),
                                            out.data_ptr(), packets.data_ptr(), 2**40, rows, 57344,
                                            8192, G, 1, 0, True, 0)
