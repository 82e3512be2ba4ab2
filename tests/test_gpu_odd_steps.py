"""An odd number of K steps (of 128 bytes) on the four-wave kernel, which walks them in pairs: the step behind the last one must add nothing,
whatever the bytes behind K hold; and row-major MX scales there, which it fetches 16 bytes of a row at a time.  Values in {0, +-0.5, +-1, +-2} and scales 2^-2 .. 2^1 (per-row scales powers of two): products are multiples
of 2^-6 and at most 16, so a sum over K <= 4480 stays below 2^17 and is exact in fp32 (23 bits): the result has to be equal to float64's.
Behind every row of A and B lie NaN codes (FP8, bf16) or sixes (FP4), behind its scales, and at the positions of the tiled layout that no block owns,
the NaN scale."""
import ctypes

import numpy as np
import pytest
import torch

import gcnasm_amd as g
import routes
from gpu_util import dev

FP8 = np.array([0x00, 0x30, 0x38, 0x40, 0xB0, 0xB8, 0xC0], np.uint8)      # 0, 0.5, 1, 2, -0.5, -1, -2
FP4 = np.array([0, 1, 2, 4, 9, 10, 12], np.uint8)
VALUE = torch.tensor([0, 0.5, 1, 2, -0.5, -1, -2], dtype=torch.float64)


def _operand(rng, rows, k, kind):
    """-> (bytes [rows, row bytes + 32] on the GPU, of which the last 32 are not the operand's; values [rows, k] float64)."""
    pick = rng.integers(0, 7, (rows, k))
    if kind == "fp4":
        c = FP4[pick]
        q, fill = (c[:, ::2] | c[:, 1::2] << 4).astype(np.uint8), 0x77
    elif kind == "bf16":
        q, fill = VALUE[torch.from_numpy(pick)].to(torch.bfloat16).view(torch.uint8).numpy(), 0xFF
    else:
        q, fill = FP8[pick], 0x7F
    store = torch.full((rows, q.shape[1] + 32), fill, dtype=torch.uint8, device="cuda")
    store[:, :q.shape[1]] = dev(np.ascontiguousarray(q))
    return store, VALUE[torch.from_numpy(pick)].cuda()


def _mx_scales(rows, k, tiled, pad):
    """-> (scale bytes on the GPU, their row stride, values [rows, k])."""
    e = (125 + (np.arange(rows)[:, None] * 3 + np.arange(k // 32)[None, :] + np.arange(rows)[:, None] // 32) % 4).astype(np.uint8)
    value = torch.from_numpy(np.exp2(e.astype(np.float64) - 127)).cuda().repeat_interleave(32, dim=1)
    store = torch.full((rows, k // 32 + pad), 255, dtype=torch.uint8, device="cuda")
    store[:, :k // 32] = dev(e)
    if not tiled:
        return store, k // 32 + pad, value
    whole = torch.full(((rows + 63) // 64 * 64, (k + 511) // 512 * 16), 255, dtype=torch.uint8, device="cuda")
    whole[:rows, :k // 32] = store[:, :k // 32]
    return g.mx_tile_scales(whole), 0, value


def _check(kind, mode, m, n, k, batch=1, pad=0):
    rng = np.random.Generator(np.random.Philox(m + n + k))
    per_byte = {"fp4": 2, "bf16": 0.5}.get(kind, 1)
    a, b = [[_operand(rng, rows, k, kind) for _ in range(batch)] for rows in (m, n)]
    if mode in (g.MX, g.MX_TILED):
        sa, sb = _mx_scales(m, k, mode == g.MX_TILED, pad), _mx_scales(n, k, mode == g.MX_TILED, pad)
        fa, fb = sa[2], sb[2]
    else:
        sa, sb = [(torch.exp2(torch.from_numpy(rng.integers(-2, 2, rows)).cuda().float()), 1, None) for rows in ((m, n) if mode == g.ROWCOL else (1, 1))]
        fa, fb = [s[0].double()[:, None] if kind != "bf16" else 1.0 for s in (sa, sb)]
    a_all, b_all = [torch.stack([o[0] for o in x]) for x in (a, b)]
    s_all = [torch.stack([s[0].flatten()] * batch) for s in (sa, sb)]
    stride = int(a_all.shape[2] * per_byte)
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        c = torch.full((batch, m, n), float("nan"), dtype=dtype, device="cuda")
        args = g.raw_gemm_args(a_all.data_ptr(), b_all.data_ptr(), c.data_ptr(), s_all[0].data_ptr(), s_all[1].data_ptr(), m, n, k, mode, c_dtype, batch,
                               stride_a=stride, stride_b=stride, stride_sfa=sa[1], stride_sfb=sb[1],
                               batch_strides=(m * stride, n * stride, m * n, s_all[0].shape[1], s_all[1].shape[1]))
        entry = {"fp4": g.lib().a4w4_gemm, "bf16": g.lib().a16w16_gemm}.get(kind, g.lib().a8w8_gemm)
        assert entry(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        for e in range(batch):
            want = (a[e][1] * fa) @ (b[e][1] * fb).T
            assert torch.equal(c[e], want.float().to(dtype)), (kind, mode, m, n, k, c_dtype, e)


# one round of ragged and of whole tiles, two tiles per workgroup, fp32 C past its own line; the fewest steps and more (the scale batches hold 8 or 4)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2790, 5111, 5), (2816, 5120, 7), (4090, 7100, 11), (2790, 5111, 13), (4350, 4200, 33)])
@pytest.mark.parametrize("kind", ["fp8", "fp4"])
def test_tiled_scales(m, n, steps, kind):
    assert routes.odd_tiled_mx_on_four_waves(m, n, steps, fp4=kind == "fp4") or (kind, steps) == ("fp4", 33)
    _check(kind, g.MX_TILED, m, n, steps * (256 if kind == "fp4" else 128))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp8", "fp4"])
def test_tiled_scales_of_a_batch(kind):
    assert routes.odd_tiled_mx_on_four_waves(2100, 2100, 5, batch=3)
    _check(kind, g.MX_TILED, 2100, 2100, 5 * (256 if kind == "fp4" else 128), batch=3)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2790, 5111, 7), (2816, 5120, 13), (4090, 7100, 17)])
@pytest.mark.parametrize("pad", [0, 4, 8])                   # scale rows of 8 bytes a step: 8 (0), 12 (4) and 0 (8) bytes past a multiple of 16
def test_mxfp4_on_row_major_scales(m, n, steps, pad):
    assert routes.f4_row_scales_on_256_tiles(m, n, steps * 256)
    _check("fp4", g.MX, m, n, steps * 256, pad=pad)


# scale rows of 4 bytes a step that start at every dword of a 16-byte piece (128, 132, 136, 140 bytes and four more); one round and two
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2300, 4099, 32), (2816, 5120, 33), (4350, 4200, 34), (4090, 7100, 33), (2300, 4099, 35)])
@pytest.mark.parametrize("pad", [0, 4])
def test_mxfp8_on_row_major_scales(m, n, steps, pad):
    assert routes.mx_row_scales_on_four_waves(steps)
    _check("fp8", g.MX, m, n, steps * 128, pad=pad)


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [32, 33])
def test_mxfp8_on_row_major_scales_of_a_batch(steps):
    _check("fp8", g.MX, 2100, 2100, steps * 128, batch=3, pad=4)


def test_rule_for_mxfp8_on_row_major_scales():
    for steps, wide in ((31, False), (32, True), (33, True)):
        assert routes.mx_row_scales_on_four_waves(steps) is wide
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, 4096, 4096, steps * 128, g.MX)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_persist")
        args.stride_sfa = (1 << 31) // 4096      # scale rows too far apart for 32-bit offsets past the end: still taken
        assert g.kernel_name(args) == "gemm_a8w8_persist"


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(2300, 4099), (4350, 4200)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.TENSOR), ("bf16", g.TENSOR)])
def test_scales_that_do_not_change_with_k(m, n, kind, mode):
    _check(kind, mode, m, n, 33 * (64 if kind == "bf16" else 128))


@pytest.mark.parametrize("m,n,steps,fp4,fp32,wide", [
    (2816, 5120, 3, False, False, False), (2816, 5120, 5, False, False, True), (2816, 5120, 9, False, True, False), (2816, 5120, 11, False, True, True),
    (2816, 5120, 11, True, True, False), (2816, 5120, 13, True, True, True), (2304, 4096, 11, False, False, False), (2304, 4096, 13, False, False, True),
    (2304, 4096, 23, True, False, False), (2304, 4096, 25, True, False, True), (2304, 4096, 31, True, True, False), (2304, 4096, 33, True, True, True),
    (8192, 2560, 31, False, False, False), (8192, 2560, 33, False, True, True), (8192, 2560, 65, True, False, False)])
def test_rule_for_tiled_scales(m, n, steps, fp4, fp32, wide):
    assert routes.odd_tiled_mx_on_four_waves(m, n, steps, fp4=fp4, fp32=fp32) is wide
    if not fp4:
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, steps * 128, g.MX_TILED, g.FP32 if fp32 else g.BF16)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_tile128")
        if wide:      # C rows too far apart for 32-bit offsets: still taken, by the 128-tile kernel
            args.stride_c = 1 << 24
            assert g.kernel_name(args) == "gemm_a8w8_tile128"


def test_rule_for_scales_that_do_not_change_with_k():
    for steps, wide in ((31, False), (33, True)):
        assert routes.odd_steps_on_four_waves(steps) is wide
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, 4096, 4096, steps * 128, g.ROWCOL)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_persist")
