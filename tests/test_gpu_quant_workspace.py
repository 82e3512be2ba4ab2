"""The per-tensor quantiser with the caller's workspace: the oracle's bytes and scale, and the same as without it, at the sizes where its launches change."""
import ctypes

import numpy as np
import pytest
import torch

import gcnasm_amd as g
from gpu_util import dev


def _call(x, ws, ws_bytes=None, offset=0):
    rows, k = x.shape
    q = torch.full((rows, k), 0xAB, dtype=torch.uint8, device="cuda")
    s = torch.full((1,), -1.0, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    wp = None if ws is None else ws.data_ptr() + offset
    assert g.lib().a8w8_quantize_ws(x.data_ptr(), rows, k, x.stride(0), q.data_ptr(), s.data_ptr(), g.TENSOR, 1, wp, ws.numel() if ws_bytes is None and ws is not None else ws_bytes or 0,
                                    stream) == 0
    return q, s


# one float4 past the single-workgroup kernel, one and two maxima more than a multiple of four, the last workgroup partly filled, all 512 maxima, several rounds
@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(1, 16388), (5, 3280), (17, 1024), (21, 1024), (163, 1380), (1024, 2052), (2048, 1024), (2048, 1028), (3000, 3004)])
def test_with_workspace(orc, rows, k):
    rng = np.random.Generator(np.random.Philox(rows + k))
    x = rng.standard_normal((rows, k), dtype=np.float32)
    x[-1, -1] = 9.0                          # the last element decides
    q0, s0 = orc.quantize(x, orc.TENSOR)
    ws = torch.full((2048,), 0xFF, dtype=torch.uint8, device="cuda")      # NaN patterns
    assert g.lib().a8w8_quantize_workspace_bytes(rows, k, g.TENSOR) == 2048
    plain = _call(dev(x), None)
    for got in (_call(dev(x), ws), plain, g.quantize(dev(x), g.TENSOR)):
        assert (got[0].cpu().numpy() == q0).all() and got[1].cpu().numpy() == s0
    # too short, off 16 bytes: not used
    before = ws.clone()
    for got in (_call(dev(x), ws, 2047), _call(dev(x), ws, 2048, offset=8)):
        assert (got[0].cpu().numpy() == q0).all() and got[1].cpu().numpy() == s0
    assert torch.equal(before, ws)


@pytest.mark.gpu
def test_special_values():
    for fill in (0.0, float("inf"), float("nan"), 1e-40):
        x = torch.zeros((64, 1024), device="cuda")
        x[40, 7] = fill
        ws = torch.zeros((2048,), dtype=torch.uint8, device="cuda")
        (q1, s1), (q0, s0) = _call(x, ws), _call(x, None)
        assert torch.equal(q1, q0) and torch.equal(s1.view(torch.int32), s0.view(torch.int32))


@pytest.mark.gpu
def test_replays(orc):
    """In a graph, replayed over new inputs: every replay against the eager result."""
    x = torch.randn((300, 1024), device="cuda")
    g.quantize(x, g.TENSOR)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        q, s = g.quantize(x, g.TENSOR)
    for i in range(4):
        x.copy_(torch.randn((300, 1024), device="cuda") * (i + 1))
        graph.replay()
        torch.cuda.synchronize()
        q0, s0 = orc.quantize(x.cpu().numpy(), orc.TENSOR)
        assert (q.cpu().numpy() == q0).all() and s.cpu().numpy() == s0


def test_sizes():
    L = g.lib()
    assert L.a8w8_quantize_workspace_bytes(4, 4096, g.TENSOR) == 0 and L.a8w8_quantize_workspace_bytes(4, 4097, g.TENSOR) == 2048
    assert L.a8w8_quantize_workspace_bytes(0, 4096, g.TENSOR) == 0 and L.a8w8_quantize_workspace_bytes(4096, 4096, g.ROWCOL) == 0
    assert L.a8w8_quantize_ws(None, 4, 4096, 4096, 0x1000, 0x2000, g.TENSOR, 1, 0x3000, 2048, None) == -1
