"""256 x 128 tiles of the 128-tile kernel: more 128 x 128 tiles than compute units, no more 256 x 128 ones, from 16 (bf16 and
MXFP4 on tiled scales: 24) K steps of 128 bytes on.  Exact operands, so the result has to be equal; step counts of every
remainder by the three stages and by the loop's two, ragged rows and columns, batches, both weight layouts.  Up to 224 rows the row
offsets of a tile (scalar, up to 224 rows on) pass the end of A's whole descriptor.  Every case is checked to take this variant."""
import numpy as np
import pytest
import torch

import gcnasm_amd as g
import routes
from gpu_util import dev
from test_gpu_a4w4_row_scales import _operand, _value
from test_gpu_random_shapes import _exact_case

pytestmark = pytest.mark.gpu


def _assert_tall(kind, m, n, k_bytes, batch=1):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert routes.tile128_variant(kind, m, n, k_bytes, batch, cus) == "256x128"


@pytest.mark.parametrize("mode", [g.TENSOR, g.ROWCOL, g.MX, g.MX_TILED])
@pytest.mark.parametrize("m,n,batch,ksteps", [(2560, 2048, 1, 16), (2177, 2064, 1, 17), (300, 4096, 4, 18), (129, 16400, 1, 16), (200, 4096, 5, 17),
                                              (224, 16400, 1, 18)])
def test_fp8(m, n, batch, ksteps, mode):
    _assert_tall("fp8", m, n, 128 * ksteps, batch)
    r = np.random.default_rng(m + n + 31 * ksteps + mode)
    _exact_case(r, "tall tiles", mode, batch, m, n, 128 * ksteps, g.FP32 if ksteps % 2 else g.BF16, shuffled=ksteps == 18)


@pytest.mark.parametrize("m,n,k,tiled", [(2560, 2048, 4096, False), (2560, 2048, 6144, True), (2177, 2063, 6400, False), (2177, 2063, 6400, True),
                                         (2049, 3584, 6144, False), (2049, 3584, 6144, True), (129, 16400, 4352, False), (200, 20480, 6400, True)])
def test_mxfp4(orc, m, n, k, tiled):
    _assert_tall("mxfp4_tiled" if tiled else "mxfp4", m, n, k // 2)
    r = np.random.default_rng(m + k)
    (qa, ea), (qb, eb) = _operand(r, m, k), _operand(r, n, k)
    ref = (_value(orc, qa, ea) @ _value(orc, qb, eb).T).float()
    sa, sb = dev(ea), dev(eb)
    if tiled:
        sa, sb = g.mx_tile_scales(sa), g.mx_tile_scales(sb)
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        got = g.gemm_a4w4(dev(qa), dev(qb), sa, sb, g.MX_TILED if tiled else g.MX, c_dtype=c_dtype)
        assert torch.equal(got, ref.to(dtype))


@pytest.mark.parametrize("m,n,k,batch", [(2560, 2048, 1536, 1), (2177, 2063, 1600, 1), (300, 4096, 1664, 4), (129, 16400, 1536, 1), (200, 4096, 1600, 5)])
def test_bf16(m, n, k, batch):
    _assert_tall("bf16", m, n, 2 * k, batch)
    gen = torch.Generator(device="cuda").manual_seed(m + k)
    a, b = (torch.randint(-4, 5, (batch, rows, k), generator=gen, device="cuda").bfloat16() for rows in (m, n))
    ref = torch.stack([x.double() @ y.double().T for x, y in zip(a, b)])
    for c_dtype, dtype in ((g.FP32, torch.float32), (g.BF16, torch.bfloat16)):
        assert torch.equal(g.gemm_a16w16(a, b, c_dtype=c_dtype), ref.to(dtype))
