"""GEMMs whose result is exact in fp32, against float64.  Values in {0, +-0.5, +-1, +-2} and scales 2^-2 .. 2^1: products are multiples of 2^-6 and at
most 16, so a sum over K <= 8448 stays below 2^18 (24 bits) and has to be equal, bit for bit.  Behind every row of A and B lie NaN codes (FP8, bf16) or sixes (FP4), behind its MX scales,
and at the positions of the tiled layout that no block owns, the NaN scale."""
import ctypes

import numpy as np
import torch

import gcnasm_amd as g
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


def check(kind, mode, m, n, k, batch=1, pad=0, shuffled=False, c_pad=0, c_shift=0, kernel=None):
    """c_pad: elements between C's rows, c_shift: in front of its first one; neither may be written, nor may the 256 rows behind C, which is as far as a tile on its
    edge reaches.  kernel: what serves FP8 operands, by type of C."""
    rng = np.random.Generator(np.random.Philox(m + n + k))
    per_byte = {"fp4": 2, "bf16": 0.5}.get(kind, 1)
    a, b = [[_operand(rng, rows, k, kind) for _ in range(batch)] for rows in (m, n)]
    if mode in (g.MX, g.MX_TILED):
        sa, sb = _mx_scales(m, k, mode == g.MX_TILED, pad), _mx_scales(n, k, mode == g.MX_TILED, pad)
        fa, fb = sa[2], sb[2]
    elif mode == g.BLOCK:
        ea, eb = [torch.from_numpy(rng.integers(-2, 2, shape)).cuda() for shape in ((k // 128, m), (n // 128, k // 128))]
        sa, sb = (torch.exp2(ea.float()), m, None), (torch.exp2(eb.float()), k // 128, None)
        fa, fb = sa[0].double().T.repeat_interleave(128, dim=1), sb[0].double().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)
    else:
        sa, sb = [(torch.exp2(torch.from_numpy(rng.integers(-2, 2, rows)).cuda().float()), 1, None) for rows in ((m, n) if mode == g.ROWCOL else (1, 1))]
        fa, fb = [s[0].double()[:, None] if kind != "bf16" else 1.0 for s in (sa, sb)]
    a_all, b_all = [torch.stack([o[0] for o in x]) for x in (a, b)]
    s_all = [torch.stack([s[0].flatten()] * batch) for s in (sa, sb)]
    stride = int(a_all.shape[2] * per_byte)
    b_batch = n * stride
    if shuffled:
        row_bytes = int(k / per_byte)
        b_all = torch.stack([g.preshuffle_b_device(o[0][:, :row_bytes].contiguous()) for o in b])
        b_batch = n * k
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        store = torch.full((c_shift + (batch * m + 256) * (n + c_pad),), -7.0, dtype=dtype, device="cuda")
        c = store[c_shift:c_shift + batch * m * (n + c_pad)].view(batch, m, n + c_pad)
        args = g.raw_gemm_args(a_all.data_ptr(), b_all.data_ptr(), c.data_ptr(), s_all[0].data_ptr(), s_all[1].data_ptr(), m, n, k, mode, c_dtype, batch,
                               stride_a=stride, stride_b=stride, stride_c=n + c_pad, stride_sfa=sa[1], stride_sfb=sb[1],
                               b_preshuffled=int(shuffled), batch_strides=(m * stride, b_batch, m * (n + c_pad), s_all[0].shape[1], s_all[1].shape[1]))
        assert kernel is None or g.kernel_name(args) == kernel[c_dtype], (m, n, k, c_dtype, g.kernel_name(args))
        entry = {"fp4": g.lib().a4w4_gemm, "bf16": g.lib().a16w16_gemm}.get(kind, g.lib().a8w8_gemm)
        assert entry(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        for e in range(batch):
            want = (a[e][1] * fa) @ (b[e][1] * fb).T
            assert torch.equal(c[e, :, :n], want.float().to(dtype)), (kind, mode, m, n, k, c_dtype, e)
        assert bool((c[:, :, n:] == -7.0).all() and (store[:c_shift] == -7.0).all() and (store[c_shift + batch * m * (n + c_pad):] == -7.0).all())
