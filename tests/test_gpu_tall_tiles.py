"""256 x 128 tiles of the 128-tile kernel: more 128 x 128 tiles than compute units, no more 256 x 128 ones, from 16 (bf16 and
MXFP4 on tiled scales: 24) K steps of 128 bytes on.  Exact operands, so the result has to be equal; step counts of every
remainder by the three stages and by the loop's two, ragged rows and columns, batches, both weight layouts."""
import numpy as np
import pytest
import torch

import gcnasm_amd as g
from gpu_util import dev
from test_gpu_a4w4_row_scales import _operand, _value
from test_gpu_random_shapes import _exact_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [g.TENSOR, g.ROWCOL, g.MX, g.MX_TILED])
@pytest.mark.parametrize("m,n,batch,ksteps", [(2560, 2048, 1, 16), (2177, 2064, 1, 17), (300, 4096, 4, 18), (129, 16400, 2, 16)])
def test_fp8(m, n, batch, ksteps, mode):
    r = np.random.default_rng(m + n + 31 * ksteps + mode)
    _exact_case(r, "tall tiles", mode, batch, m, n, 128 * ksteps, g.FP32 if ksteps % 2 else g.BF16, shuffled=ksteps == 18)


@pytest.mark.parametrize("m,n,k", [(2560, 2048, 4096), (2177, 2063, 6400), (2049, 3584, 6144)])
@pytest.mark.parametrize("tiled", [False, True])
def test_mxfp4(orc, m, n, k, tiled):
    r = np.random.default_rng(m + k)
    (qa, ea), (qb, eb) = _operand(r, m, k), _operand(r, n, k)
    ref = (_value(orc, qa, ea) @ _value(orc, qb, eb).T).float()
    sa, sb = dev(ea), dev(eb)
    if tiled:
        sa, sb = g.mx_tile_scales(sa), g.mx_tile_scales(sb)
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        got = g.gemm_a4w4(dev(qa), dev(qb), sa, sb, g.MX_TILED if tiled else g.MX, c_dtype=c_dtype)
        assert torch.equal(got, ref.to(dtype))


@pytest.mark.parametrize("m,n,k,batch", [(2560, 2048, 1536, 1), (2177, 2063, 1600, 1), (300, 4096, 1664, 4)])
def test_bf16(m, n, k, batch):
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    a, b = (torch.randint(-4, 5, (batch, rows, k), generator=gen, device="cuda").bfloat16() for rows in (m, n))
    ref = torch.stack([x.double() @ y.double().T for x, y in zip(a, b)])
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        assert torch.equal(g.gemm_a16w16(a, b, c_dtype=c_dtype), ref.to(dtype))
