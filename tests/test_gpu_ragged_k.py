"""K that is no multiple of the 128-byte K step, on the 128-tile kernel's partial last step: every staging variant, remainders
of one piece to seven, step counts around the stage counts; NaN codes in the padding behind every row must never be seen.
Small integers with power-of-two scales are exact in fp32; on normal data the fp32 result has to stay within 1e-7 of
sum |a||b|s of the float64 value (ten times what fp32 sums on the bf16 MFMA, and sequential ones, were measured to differ by
over K = 4096; the FP8 MFMA differs by 1.6e-6)."""
import numpy as np
import pytest
import torch

import gcnasm_amd as g
import oracle
from gpu_util import exact64

pytestmark = pytest.mark.gpu


def _padded(x, fill, pad=16):
    whole = torch.full(x.shape[:-1] + (x.shape[-1] + pad,), fill, dtype=x.dtype, device="cuda")
    whole[..., : x.shape[-1]] = x.cuda()
    return whole[..., : x.shape[-1]]


# (m, n): 128 x 128 tiles on four stages (small grid, few steps), on two stages (a large grid), 128 x 64 tiles (long K)
@pytest.mark.parametrize("m,n,k,batch", [(300, 391, 144, 1), (300, 391, 240, 2), (300, 391, 624, 1), (257, 384, 1136, 1),
                                         (2177, 2061, 400, 1), (129, 1000, 2000, 1), (1, 4100, 2064, 1), (700, 260, 48, 9)])
@pytest.mark.parametrize("mode", [g.TENSOR, g.ROWCOL, "bf16"])
def test_partial_last_step_is_exact(m, n, k, batch, mode):
    r = np.random.default_rng(m + n + k)
    a, b = (r.integers(-4, 5, (batch, rows, k)).astype(np.float32) for rows in (m, n))
    for cdt in (torch.bfloat16, torch.float32):
        c = torch.full((batch, m, n + 8), 7.0, dtype=cdt, device="cuda")
        if mode == "bf16":
            want = np.einsum("bmk,bnk->bmn", a, b)
            da, db = (_padded(torch.from_numpy(x).to(torch.bfloat16), float("nan")) for x in (a, b))
            g.gemm_a16w16(da if batch > 1 else da[0], db if batch > 1 else db[0], c=(c if batch > 1 else c[0])[..., :n])
        else:
            shape = (lambda rows: (batch, rows if mode == g.ROWCOL else 1))
            sa, sb = (np.exp2(r.integers(-2, 3, shape(rows))).astype(np.float32) for rows in (m, n))
            want = np.einsum("bmk,bnk->bmn", a, b) * sa[:, :, None] * sb[:, None, :]
            da, db = (_padded(torch.from_numpy(oracle.encode(x)), 0x7F) for x in (a, b))
            args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, k, mode, batch=batch)
            assert g.kernel_name(args) == "gemm_a8w8_tile128"
            ts = [torch.from_numpy(s).cuda() for s in (sa, sb)]
            pick = (lambda t: t) if batch > 1 else (lambda t: t[0])
            g.gemm(pick(da), pick(db), pick(ts[0]), pick(ts[1]), mode, c=pick(c)[..., :n])
        torch.cuda.synchronize()
        ref = torch.from_numpy(want.astype(np.float32)).to(cdt).float().numpy()
        assert (c[..., :n].float().cpu().numpy() == ref).all()
        assert (c[..., n:].float() == 7.0).all()


def test_partial_last_step_keeps_fp32_sums(orc):
    m, n, k = 200, 300, 2000
    r = np.random.default_rng(5)
    a, b = (oracle.encode((r.standard_normal((rows, k)) * 100).astype(np.float32)) for rows in (m, n))
    sa, sb = np.ones(m, np.float32), np.ones(n, np.float32)
    got = g.gemm(*(torch.from_numpy(x).cuda() for x in (a, b, sa, sb)), g.ROWCOL, c_dtype=g.FP32).cpu().numpy()
    exact, mag = exact64(orc, a, b, sa, sb, g.ROWCOL)
    assert (np.abs(got - exact) <= 1e-7 * mag).all()


@pytest.mark.parametrize("side", ["a", "b"])
def test_partial_last_step_at_the_end_of_two_gigabytes(side):
    """A matrix that ends 16 bytes below 2 GiB: the pieces past K of its last row lie beyond 2^31, where a lane offset with bit 31
    on top, plus the step's scalar offset, would wrap to the matrix's first bytes.  Those are NaN codes here: row 0 is NaN, and
    no other row may be."""
    rows, stride, k, other = 3, 1073741680, 272, 64
    assert (rows - 1) * stride + k == 2 ** 31 - 16
    r = np.random.default_rng(9)
    x, y = (r.integers(-4, 5, (m, k)).astype(np.float32) for m in (rows, other))
    whole = torch.empty(2 ** 31, dtype=torch.uint8, device="cuda")
    long = whole.as_strided((rows, k), (stride, 1))
    long.copy_(torch.from_numpy(oracle.encode(x)))
    long[0, :16] = 0x7F
    short = torch.from_numpy(oracle.encode(y)).cuda()
    one = torch.ones(1, device="cuda")
    a, b = (long, short) if side == "a" else (short, long)
    assert g.kernel_name(g.raw_gemm_args(a.data_ptr(), b.data_ptr(), 1 << 12, 1 << 12, 1 << 12, a.shape[0], b.shape[0], k, g.TENSOR,
                                         stride_a=a.stride(0), stride_b=b.stride(0))) == "gemm_a8w8_tile128"
    got = g.gemm(a, b, one, one, g.TENSOR, c_dtype=g.FP32)
    got = (got if side == "a" else got.T).cpu().numpy()
    assert np.isnan(got[0]).all()
    assert (got[1:] == x[1:] @ y.T).all()
