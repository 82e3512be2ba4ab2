"""Tensors that the kernels would misread, or read past their end, are refused before any launch: elements of another size, columns apart, too few bytes or
scales, host memory.  On the CPU by the functions' own statements; on the GPU the compiled path (csrc/binding.cpp) has to decline the same tensors."""
import pytest
import torch

import gcnasm_amd as g
from gcnasm_amd import api


def _forms(device):
    """(function, arguments, exception) over tensors on `device`; where it is the host, what is right otherwise is refused for that."""
    def t(*shape, dtype=torch.uint8):
        return torch.zeros(shape, dtype=dtype, device=device)
    x = t(256, 512, dtype=torch.float32)
    wrong_rows = [(x.bfloat16(), TypeError), (x.half(), TypeError), (x.double(), TypeError), (x.int(), TypeError), (x.T, ValueError), (x[:, ::2], ValueError)]
    for mode in (g.TENSOR, g.ROWCOL, g.BLOCK, g.MX, g.MX_TILED):
        yield from ((g.quantize, (bad, mode), e) for bad, e in wrong_rows)
    for tiled in (False, True):
        yield from ((g.quantize_mxfp4, (bad, tiled), e) for bad, e in wrong_rows)
    yield from ((g.cvt_f32_to_e4m3, (bad,), TypeError) for bad in (x.bfloat16(), x.half(), x.double(), x.int()))
    yield from ((g.cvt_e4m3_to_f32, (bad,), TypeError) for bad in (x, x.bfloat16(), x.int()))
    # GEMMs: a, b, scales, c
    a, b, f, rows = t(48, 512), t(256, 512), t(4096, dtype=torch.float32), t(48, dtype=torch.float32)
    wide = t(48, 1024)
    for bad_a, bad_b, e in ((a.float(), b, TypeError), (a, b.bfloat16(), TypeError), (wide[:, ::2], b, ValueError), (a, t(512, 256).T, ValueError), (a, b[:, :384], ValueError)):
        yield g.gemm, (bad_a, bad_b, f, f, g.ROWCOL), e
        yield g.gemm_blockscale, (bad_a, bad_b, f, f), e
        yield g.gemm_a4w4, (bad_a, bad_b, t(1 << 16), t(1 << 16)), e
    yield g.gemm_a16w16, (a, b), TypeError
    yield g.gemm_a16w16, (a.bfloat16(), b), TypeError
    yield g.gemm_a16w16, (a.bfloat16(), b.bfloat16()[:, :384]), ValueError
    flat = t(256 * 512)
    for short in (flat[:-1], flat[::2], t(256, 1024)[:, :512]):
        yield g.gemm, (a, short, f, f, g.ROWCOL, None, g.BF16, 256), ValueError
        yield g.flatmm, (a, short, f, f, 256), ValueError
        yield g.flatmm_a16w16, (a.bfloat16(), short, 256), ValueError
        yield g.flatmm_a4w4, (a, short, t(1 << 16), t(1 << 16), 256), ValueError
        yield g.gemm_a4w4, (a, short, t(1 << 16), t(1 << 16), g.MX_TILED, None, g.BF16, 256), ValueError
    for mode, need_a, need_b in ((g.MX, 48 * 32, 256 * 32), (g.MX_TILED, 2048, 8192)):
        for sa, sb, e in ((t(need_a - 1), t(need_b), ValueError), (t(need_a), t(need_b - 1), ValueError), (t(need_a, dtype=torch.float32), t(need_b), TypeError),
                          (t(need_a), t(need_b, dtype=torch.int16), TypeError), (t(2 * need_a)[::2], t(need_b), ValueError)):
            yield g.gemm_a4w4, (a, b, sa, sb, mode), e
            if mode == g.MX_TILED:
                yield g.flatmm_a4w4, (a, flat, sa, sb, 256), e
    for c, e in ((t(48, 512, dtype=torch.bfloat16)[:, ::2], ValueError), (t(48, 256, dtype=torch.half), TypeError), (t(48, 255, dtype=torch.float32), ValueError),
                 (torch.zeros(48, 256), ValueError)):
        yield g.gemm, (a, b, rows, f, g.ROWCOL, c), e
        yield g.gemm_a4w4, (a, b, t(2048), t(8192), g.MX_TILED, c), e
    # weights and scales that are laid out once
    yield from ((g.preshuffle_b_device, (bad,), e) for bad, e in ((b.float(), TypeError), (b[:, :256], ValueError), (b.T, ValueError)))
    yield from ((g.mx_tile_scales, (bad,), e) for bad, e in ((b.float(), TypeError), (b.T, ValueError), (b[:, ::2], ValueError)))
    yield g.mx_tile_scales, (t(64, 16), t(1023)), ValueError
    yield g.mx_tile_scales_ab, (t(64, 16), t(64, 15)), ValueError
    yield g.mx_tile_scales_ab, (t(64, 16), t(16, 64).T), ValueError
    # host memory
    if device != "cpu":
        return
    for function, args in ((g.quantize, (x, g.ROWCOL)), (g.quantize_mxfp4, (x,)), (g.cvt_f32_to_e4m3, (x,)), (g.cvt_e4m3_to_f32, (a,)), (g.gemm, (a, b, f, f, g.ROWCOL)),
                           (g.gemm_a16w16, (a.bfloat16(), b.bfloat16())), (g.gemm_a4w4, (a, b, t(2048), t(8192))), (g.flatmm, (a, flat, f, f, 256)),
                           (g.flatmm_a4w4, (a, flat, t(2048), t(8192), 256)), (g.preshuffle_b_device, (b,)), (g.mx_tile_scales, (b,)), (g.mx_tile_scales_ab, (b, b))):
        yield function, args, ValueError


def test_refused_on_the_host():
    forms = list(_forms("cpu"))
    assert len(forms) > 100
    for i, (function, args, e) in enumerate(forms):
        with pytest.raises((e, ValueError)):      # (or for the first tensor's being on the host)
            function(*args)
            pytest.fail(f"{i} {function.__name__}")


@pytest.mark.gpu
def test_refused_on_the_gpu(monkeypatch):
    served = []
    api._connect()
    for name in ("_fast_gemm", "_fast_quantize", "_fast_quantize_mxfp4", "_fast_encode", "_fast_decode"):
        def seen(*args, fast=getattr(api, name)):
            served.append(fast(*args))
            return served[-1]
        monkeypatch.setattr(api, name, seen)
    for i, (function, args, e) in enumerate(_forms("cuda")):
        with pytest.raises(e):
            function(*args)
            pytest.fail(f"{i} {function.__name__}")
    assert len(served) > 80 and all(r is None for r in served)


@pytest.mark.gpu
def test_still_taken():
    """One-byte and two-byte types other than uint8 and bfloat16 as bits, and buffers larger than what is read."""
    def bits(t, dtype):
        return t.view(dtype)
    x, w = torch.randn(48, 512, device="cuda"), torch.randn(256, 512, device="cuda")
    (a, sa), (b, sb) = g.quantize(x, g.ROWCOL), g.quantize(w, g.ROWCOL)
    want = g.gemm(a, b, sa, sb, g.ROWCOL)
    for dtype in (torch.float8_e4m3fn, torch.int8):
        assert torch.equal(g.gemm(bits(a, dtype), bits(b, dtype), sa, sb, g.ROWCOL), want)
        assert torch.equal(g.cvt_e4m3_to_f32(bits(a, dtype)), g.cvt_e4m3_to_f32(a))
    assert torch.equal(g.gemm(a[:, :384], b, sa, sb, g.ROWCOL), g.gemm(a[:, :384], b[:, :384], sa, sb, g.ROWCOL))
    flat = torch.cat([g.preshuffle_b_device(b), torch.zeros(512, dtype=torch.uint8, device="cuda")])
    assert torch.equal(g.flatmm(a, flat, sa, sb, 256), g.flatmm(a, flat[:-512], sa, sb, 256))
    (a, sa), (b, sb) = g.quantize_mxfp4(x, True), g.quantize_mxfp4(w, True)
    assert torch.equal(g.gemm_a4w4(a, b, bits(sa, torch.int8), bits(sb, torch.int8)), g.gemm_a4w4(a, b, sa, sb))
    one = torch.randn(40, 1, device="cuda").T      # a single row whose column stride is 1 and row stride is not its length
    assert torch.equal(g.cvt_f32_to_e4m3(one), g.cvt_f32_to_e4m3(one.clone()))


@pytest.mark.gpu
def test_strides_past_an_int():
    """2^32 elements between rows or batch entries would arrive at the library as 0, i.e. as the first row or entry again."""
    x = torch.empty((1 << 32) + 512, device="cuda").as_strided((2, 512), (1 << 32, 1))      # 16 GiB, of which nothing is read
    for quantize in (lambda: g.quantize(x, g.ROWCOL), lambda: g.quantize_mxfp4(x)):
        with pytest.raises(g.A8W8Error, match="-7"):
            quantize()
    del x
    a = torch.empty((1 << 32) + 16 * 512, dtype=torch.uint8, device="cuda")
    b, s = torch.zeros((256, 512), dtype=torch.uint8, device="cuda"), torch.ones(512, device="cuda")
    for batched in (a.as_strided((2, 16, 512), (1 << 32, 512, 1)), a.as_strided((2, 512), (1 << 32, 1))):
        with pytest.raises(g.A8W8Error, match="-7"):
            g.gemm(batched, b, s, s, g.ROWCOL)
    assert g.gemm(a.as_strided((1, 16, 512), (1 << 32, 512, 1)), b, s, s, g.ROWCOL).shape == (1, 16, 256)      # (no second entry)
    e = torch.zeros(1 << 14, dtype=torch.uint8, device="cuda")
    with pytest.raises(g.A8W8Error, match="-7"):
        g.gemm_a4w4(a.as_strided((2, 512), (1 << 31, 1)), b, e, e)


def test_ints():
    api._check_ints("here", 0, (1 << 31) - 1)
    with pytest.raises(g.A8W8Error, match="-7"):
        api._check_ints("here", 5, 1 << 31)
