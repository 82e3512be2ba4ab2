"""The compiled path of the public functions (csrc/binding.cpp) against their own statements in api.py, which serve whatever it declines: the same outputs
bit for bit, or the same exception with the same text, over the forms that the functions take and refuse."""
import pytest
import torch

import gcnasm_amd as g
from gcnasm_amd import api

FAST = ("_fast_gemm", "_fast_quantize", "_fast_quantize_mxfp4", "_fast_encode", "_fast_decode")


def _rand(*shape, **kw):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(sum(shape))
    return torch.randn(shape, generator=gen, device="cuda", **kw)


class Sub(torch.Tensor):
    pass


def _quantized(mode, rows, k, weight=False, batch=0):
    pairs = [g.quantize(_rand(rows, k) + i, mode, group_rows=128 if weight and mode == g.BLOCK else 1) for i in range(max(batch, 1))]
    return (torch.stack([p[0] for p in pairs]), torch.stack([p[1] for p in pairs])) if batch else pairs[0]


def _gemm_forms():
    for mode in (g.TENSOR, g.ROWCOL, g.BLOCK, g.MX, g.MX_TILED):
        (a, sa), (b, sb) = _quantized(mode, 48, 512), _quantized(mode, 256, 512, True)
        yield g.gemm, (a, b, sa, sb, mode), {}
        yield g.gemm, (a, b, sa, sb, mode), dict(c_dtype=g.FP32)
        yield g.gemm, (a, b, sa, sb, mode), dict(c=torch.full((48, 256 + 8), 3.0, dtype=torch.bfloat16, device="cuda")[:, :256])
        yield g.gemm, (a, b, sa, sb, mode), dict(c=torch.zeros((48, 256), device="cuda"), c_dtype=g.BF16)
        yield g.gemm, (a, g.preshuffle_b_device(b), sa, sb, mode), dict(n=256)
        wide = torch.zeros((48, 512 + 64), dtype=torch.uint8, device="cuda")
        wide[:, :512] = a
        yield g.gemm, (wide[:, :512], b, sa, sb, mode), {}
        yield g.gemm, (a, b, sa.cpu(), sb, mode), {}
        yield g.gemm, (a, b, sa.to(torch.float64), sb, mode), {}
        yield g.gemm, (a, b, sa.flatten()[:-1] if sa.numel() > 1 else sa[:0], sb, mode), {}
        yield g.gemm, (a, b, sa, sb.flatten()[:-1] if sb.numel() > 1 else sb[:0], mode), {}
        (a3, sa3), (b3, sb3) = _quantized(mode, 40, 512, batch=3), _quantized(mode, 256, 512, True, batch=3)
        yield g.gemm, (a3, b3, sa3, sb3, mode), {}
        yield g.gemm, (a3, b, sa3, sb, mode), {}
        yield g.gemm, (a3, b, sa3, sb3, mode), {}
        yield g.gemm, (a3, b3[:2], sa3, sb3, mode), {}
        yield g.gemm, (a3, g.preshuffle_b_device(b), sa3, sb, mode), dict(n=256)
        yield g.gemm, (a3[:1], b3[:1], sa3[:1].contiguous(), sb3[:1].contiguous(), mode), {}
        yield g.gemm, (a3, b3, sa3, sb3, mode), dict(c=torch.zeros((3, 40, 256), device="cuda"))
        yield g.gemm, (a, b3, sa, sb3, mode), {}
    (a, sa), (b, sb) = _quantized(g.ROWCOL, 48, 512), _quantized(g.ROWCOL, 256, 512)
    yield g.gemm, (a, b, sa, sb, 9), {}
    yield g.gemm, (a, b, sa, sb, g.ROWCOL), dict(c_dtype=5)
    yield g.gemm, (a.cpu(), b, sa, sb, g.ROWCOL), {}
    yield g.gemm, (a[:, ::2], b[:, :256], sa, sb, g.ROWCOL), {}
    yield g.gemm, (a.T, b, sa, sb, g.ROWCOL), {}
    yield g.gemm, (a[0], b, sa, sb, g.ROWCOL), {}
    yield g.gemm, (a, b, sa[::2], sb, g.ROWCOL), {}
    yield g.gemm, (a[:0], b, sa, sb, g.ROWCOL), {}
    yield g.gemm, (a, b, sa, sb, g.ROWCOL), dict(c=torch.zeros((48, 256), dtype=torch.float16, device="cuda"))
    yield g.gemm, (a, b, sa, sb, g.ROWCOL), dict(c=torch.zeros((256, 48), device="cuda").T)
    yield g.gemm, (a, b, sa, sb, g.ROWCOL), dict(c=torch.zeros((48, 255), device="cuda"))
    yield g.gemm, (a.as_subclass(Sub), b, sa, sb, g.ROWCOL), {}
    yield g.gemm, (a, torch.nn.Parameter(b, requires_grad=False), sa, sb.clone().requires_grad_(), g.ROWCOL), {}
    yield g.gemm, (a, g.preshuffle_b_device(b), sa, sb, g.ROWCOL), dict(n=250)
    yield g.flatmm, (a, g.preshuffle_b_device(b), sa, sb, 256), {}
    yield g.flatmm, (a, g.preshuffle_b_device(b), sa, sb, 256), dict(c_dtype=g.FP32)
    yield g.flatmm, (_quantized(g.ROWCOL, 200, 512)[0], g.preshuffle_b_device(b), _quantized(g.ROWCOL, 200, 512)[1], sb, 256), {}
    (a, sa), (b, sb) = _quantized(g.BLOCK, 48, 512), _quantized(g.BLOCK, 256, 512, True)
    yield g.gemm_blockscale, (a, b, sa, sb), {}
    yield g.gemm_blockscale, (a, b, sa, sb), dict(c_dtype=g.BF16)
    yield g.gemm_blockscale, (a[:, :448], b[:, :448], sa, sb), {}
    x, w = _rand(48, 512).bfloat16(), _rand(256, 512).bfloat16()
    yield g.gemm_a16w16, (x, w), {}
    yield g.gemm_a16w16, (x, w), dict(c_dtype=g.FP32)
    yield g.gemm_a16w16, (torch.stack([x] * 3), torch.stack([w] * 3)), {}
    yield g.gemm_a16w16, (torch.stack([x] * 3), w), {}
    yield g.gemm_a16w16, (x, g.preshuffle_b_bf16_device(w)), dict(n=256)
    yield g.gemm_a16w16, (torch.stack([x] * 2), g.preshuffle_b_bf16_device(w)), dict(n=256)
    yield g.flatmm_a16w16, (x, g.preshuffle_b_bf16_device(w), 256), {}
    yield g.flatmm_a16w16, (x[:, :500], g.preshuffle_b_bf16_device(w), 256), {}
    for tiled in (False, True):
        (a, sa), (b, sb) = g.quantize_mxfp4(_rand(48, 512), tiled=tiled), g.quantize_mxfp4(_rand(256, 512), tiled=tiled)
        yield g.gemm_a4w4, (a, b, sa, sb, g.MX_TILED if tiled else g.MX), {}
        yield g.gemm_a4w4, (a, b, sa, sb, g.MX_TILED if tiled else g.MX), dict(c_dtype=g.FP32, c=torch.zeros((48, 256 + 16), device="cuda")[:, :256])
    yield g.gemm_a4w4, (a, b, sa, sb, g.ROWCOL), {}
    yield g.gemm_a4w4, (a, g.preshuffle_b_device(b), sa, sb), dict(n=256)
    yield g.flatmm_a4w4, (a, g.preshuffle_b_device(b), sa, sb, 256), {}
    yield g.flatmm_a4w4, (a, g.preshuffle_b_device(b), sa, sb, 256), dict(c=torch.zeros((48, 128), device="cuda"))


def _other_forms():
    x = _rand(40, 512)
    for mode in (g.TENSOR, g.ROWCOL, g.BLOCK, g.MX, g.MX_TILED):
        for t in (x, x[:, :384], x[:, :100], x[:0], x[0], _rand(300, 1024), torch.nn.Parameter(x), x.as_subclass(Sub), x[::2]):
            yield g.quantize, (t, mode), {}
    yield g.quantize, (_rand(256, 512), g.BLOCK, 128), {}
    yield g.quantize, (x, g.BLOCK, 128), {}
    yield g.quantize, (x, g.BLOCK, 64), {}
    yield g.quantize, (x, 7), {}
    for t in (x, x[:, :384], x[:, :100], x[:0], x[0], x[::2]):
        yield g.quantize_mxfp4, (t,), {}
        yield g.quantize_mxfp4, (t,), dict(tiled=True)
    for t in (x, x[0], x[:, ::2], x.T, x[:0], _rand(7), torch.tensor(3.0, device="cuda")):
        for dialect in (g.OCP, g.FNUZ, 3):
            yield g.cvt_f32_to_e4m3, (t, dialect), {}
            yield g.cvt_f32_to_e4m3, (t,), dict(dialect=dialect, clamp240=True)
            yield g.cvt_e4m3_to_f32, ((t * 50).to(torch.int32).to(torch.uint8), dialect), {}


def _ordinary(f, args, kw):
    """What csrc/binding.cpp is for: torch's own tensors in GPU memory, contiguous ones for the conversions, and no batch of b alone."""
    tensors = [t for t in (*args, kw.get("c")) if isinstance(t, torch.Tensor)]
    if not all(type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda for t in tensors):
        return False
    return args[0].is_contiguous() if f in (g.cvt_f32_to_e4m3, g.cvt_e4m3_to_f32) else f is not g.gemm or args[1].dim() <= args[0].dim()


def _recorded(patch):
    """Answers of the compiled path from here on, None where it declines."""
    answers = []
    for name in FAST:
        def call(*args, fast=getattr(api, name)):
            answers.append(fast(*args))
            return answers[-1]
        patch.setattr(api, name, call)
    return answers


def _outcome(f, args, kw):
    kw = dict(kw)
    given = kw.get("c")
    if given is not None:
        kw["c"] = given.clone() if given.is_contiguous() else given
        kw["c"].fill_(7)
    try:
        out = f(*args, **kw)
    except Exception as e:
        return type(e), str(e)
    if given is not None:
        assert out is kw["c"]
    return [t.clone() for t in (out if isinstance(out, tuple) else (out,))]


@pytest.mark.gpu
@pytest.mark.parametrize("forms", [_gemm_forms, _other_forms], ids=lambda f: f.__name__)
def test_same_as_the_statements_of_the_functions(forms, monkeypatch):
    g.quantize(_rand(4, 128), g.ROWCOL)      # connects
    served, declined = set(), 0
    for i, (f, args, kw) in enumerate(forms()):
        with monkeypatch.context() as patch:
            answers = _recorded(patch)
            fast = _outcome(f, args, kw)
        assert len(answers) == 1, (i, f.__name__)
        with monkeypatch.context() as patch:
            for name in FAST:
                patch.setattr(api, name, lambda *a: None)
            slow = _outcome(f, args, kw)
        if isinstance(slow, tuple):
            assert fast == slow, (i, f.__name__, kw, fast, slow)
        else:
            assert (answers[0] is not None) == _ordinary(f, args, kw), (i, f.__name__, kw)
            if answers[0] is None:
                declined += 1
            else:
                served.add(i)
            for u, v in zip(fast, slow):
                assert type(u) is type(v) and u.dtype == v.dtype and u.shape == v.shape and u.stride() == v.stride() and torch.equal(u.view(torch.uint8) if u.dim() else u, v.view(torch.uint8) if v.dim() else v), (i, f.__name__, kw)
    assert len(served) >= 40 and declined > 0


@pytest.mark.gpu
def test_on_the_current_stream_and_under_modes(monkeypatch):
    x = _rand(64, 1024)
    want = g.quantize(x, g.ROWCOL)
    answers = _recorded(monkeypatch)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        y = x * 1.0
        got = g.quantize(y, g.ROWCOL)
    s.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with torch.inference_mode():
        q, _ = g.quantize(x, g.ROWCOL)
        assert q.is_inference()
    assert len(answers) == 2 and all(r is not None for r in answers)
    with torch.device("cpu"):                # a function mode: the functions' own statements
        assert torch.equal(g.quantize(x, g.ROWCOL)[0], want[0])
    seen = []

    class Log(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Log():
        assert torch.equal(g.quantize(x, g.ROWCOL)[0], want[0])
    assert torch.ops.aten.empty.memory_format in seen      # allocations go through the mode
    assert len(answers) == 4 and answers[2] is None and answers[3] is None
    with pytest.raises(Exception):           # no address behind a batched tensor
        torch.vmap(lambda t: g.quantize(t, g.ROWCOL)[0])(torch.stack([x, x]))


def test_declines_what_is_not_an_ordinary_gpu_tensor():
    api._connect()
    x = torch.zeros(4, 128)
    assert api._fast_quantize(x, g.ROWCOL, 1) is None and api._fast_encode(x, 0, 0) is None and api._fast_decode(x, 0) is None
    assert api._fast_quantize(None, g.ROWCOL, 1) is None and api._fast_quantize(x, g.ROWCOL) is None and api._fast_quantize_mxfp4(x, "yes") is None
    assert api._fast_gemm(0, x, x, x, x, g.ROWCOL, None, 0, None) is None and api._fast_gemm() is None
    assert api._done(None, "x") is None and api._done(x, "x") is x
    with pytest.raises(g.A8W8Error):
        api._done(-3, "x")
