"""MXFP4 with row-major scales past two 128-tiles per compute unit: the four-wave kernel where the scale rows take its 16-byte
loads and its rounds pay (f4_row_scales_on_256_tiles of routes.hpp), the 128-tile kernel elsewhere.  Values in {0, +-0.5, +-1, +-2}, scales 2^-2 .. 2^1: products are multiples of 2^-6 and at
most 16, so a sum over K <= 2048 stays below 2^15 and is exact in fp32 (21 bits): the result has to be equal."""
import ctypes

import numpy as np
import pytest
import torch

import gcnasm_amd as g
import routes
from gpu_util import dev

pytestmark = pytest.mark.gpu

CODES = np.array([0, 1, 2, 4, 9, 10, 12], np.uint8)          # 0, 0.5, 1, 2, -0.5, -1, -2


def _operand(rng, rows, k):
    c = CODES[rng.integers(0, len(CODES), (rows, k))]
    q = (c[:, ::2] | c[:, 1::2] << 4).astype(np.uint8)
    s = (125 + (np.arange(rows)[:, None] * 3 + np.arange(k // 32)[None, :] + np.arange(rows)[:, None] // 32) % 4).astype(np.uint8)
    return q, s


def _value(orc, q, s):
    return torch.from_numpy(orc.e2m1_decode_packed(q).astype(np.float64) * np.exp2(s.astype(np.float64) - 127).repeat(32, axis=1)).cuda()


# whole tiles, ragged edges in both directions
@pytest.mark.parametrize("m,n,k", [(4096, 4096, 512), (4350, 2311, 1024), (2049, 4097, 1536), (6145, 2050, 2048), (4200, 4100, 768)])
@pytest.mark.parametrize("pad", [0, 16, 4])                  # bytes between scale rows; 4 (and k = 768): the 128-tile kernel
def test_exact_against_float64(orc, m, n, k, pad):
    rng = np.random.Generator(np.random.Philox(m + k + pad))
    (qa, ea), (qb, eb) = _operand(rng, m, k), _operand(rng, n, k)
    ref = _value(orc, qa, ea) @ _value(orc, qb, eb).T
    stride = k // 32 + pad
    sa, sb = (torch.full((e.shape[0], stride), 200, dtype=torch.uint8, device="cuda") for e in (ea, eb))
    sa[:, :k // 32], sb[:, :k // 32] = dev(ea), dev(eb)
    a, b = dev(qa), dev(qb)
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        c = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        args = g.raw_gemm_args(a.data_ptr(), b.data_ptr(), c.data_ptr(), sa.data_ptr(), sb.data_ptr(), m, n, k, g.MX, c_dtype,
                               stride_sfa=stride, stride_sfb=stride)
        assert g.lib().a4w4_gemm(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        assert torch.equal(c, ref.to(torch.float32).to(dtype))


def test_batch_with_padded_scale_sets(orc):
    """Three problems in one launch, scale sets 48 bytes apart more than they need."""
    _batch_with_padded_scale_sets(orc, 2100, 2100, 1024, 3)


def _batch_with_padded_scale_sets(orc, m, n, k, batch):
    rng = np.random.Generator(np.random.Philox(5))
    ops = [(_operand(rng, m, k), _operand(rng, n, k)) for _ in range(batch)]
    a, b = (torch.stack([dev(o[i][0]) for o in ops]) for i in range(2))
    per = [m * (k // 32) + 48, n * (k // 32) + 48]
    s = [torch.zeros(batch, per[i], dtype=torch.uint8, device="cuda") for i in range(2)]
    for e, o in enumerate(ops):
        for i in range(2):
            s[i][e, :o[i][1].size] = dev(o[i][1]).flatten()
    c = torch.zeros((batch, m, n), device="cuda")
    args = g.raw_gemm_args(a.data_ptr(), b.data_ptr(), c.data_ptr(), s[0].data_ptr(), s[1].data_ptr(), m, n, k, g.MX, g.FP32, batch,
                           batch_strides=(m * k, n * k, m * n, per[0], per[1]))
    assert g.lib().a4w4_gemm(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    for e, o in enumerate(ops):
        assert torch.equal(c[e], (_value(orc, *o[0]) @ _value(orc, *o[1]).T).float())


# the four-wave kernel: two to nine pairs of K steps (the scale batches hold two), whole and ragged tiles, one round and two
@pytest.mark.parametrize("m,n,k,fp32", [(4096, 4096, 1024, False), (3900, 3850, 1536, False), (3900, 3850, 2048, True), (6145, 2050, 2560, True),
                                        (3001, 7000, 3072, False), (2049, 4097, 4096, True), (2049, 4097, 4608, False)])
@pytest.mark.parametrize("pad", [0, 16])
def test_four_wave_kernel_is_exact(orc, m, n, k, fp32, pad):
    assert routes.f4_row_scales_on_256_tiles(m, n, k, fp32=fp32)
    test_exact_against_float64(orc, m, n, k, pad)


def test_four_wave_kernel_batch(orc):
    m, n, k, batch = 2100, 2100, 2048, 3
    assert routes.f4_row_scales_on_256_tiles(m, n, k, batch, fp32=True)
    _batch_with_padded_scale_sets(orc, m, n, k, batch)
