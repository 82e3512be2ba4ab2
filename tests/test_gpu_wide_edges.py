"""Where the four-wave kernel's tiles meet the edges of C, and C rows that start on dwords only: tiles that end with the matrix in either direction go through
a descriptor that ends there, columns past n are left out by groups of 64 (bf16) or 32 (fp32), and nothing outside C may be written.  Exact results
(exact_gemm.py)."""
import pytest

import gcnasm_amd as g
import routes
from exact_gemm import check

pytestmark = pytest.mark.gpu

WIDE = {g.BF16: "gemm_a8w8_wide", g.FP32: "gemm_a8w8_wide"}
SMALL = {g.BF16: "gemm_a8w8_tile128", g.FP32: "gemm_a8w8_tile128"}      # badly filled rounds, or few steps of an odd number: the same edges there
BF16_WIDE = {g.BF16: "gemm_a8w8_wide", g.FP32: "gemm_a8w8_tile128"}


# one and two rounds of tiles; n that ends on 128, 64, 32, 16, 4 columns, on one; m one row into a tile, one short of it
@pytest.mark.parametrize("m,n", [(2816, 4736), (2561, 4672), (2815, 4704), (4351, 4240), (2700, 4700), (2305, 4097), (4200, 4224), (129, 33024)])
@pytest.mark.parametrize("kind,mode,k", [("fp8", g.ROWCOL, 512), ("fp8", g.MX_TILED, 768), ("fp8", g.MX_TILED, 2816), ("bf16", g.TENSOR, 256), ("fp4", g.MX_TILED, 1024)], ids=lambda v: str(v))
def test_edges(m, n, kind, mode, k):
    kernel = WIDE
    if k == 768:
        kernel = {(4351, 4240): SMALL, (4200, 4224): SMALL, (2305, 4097): BF16_WIDE, (129, 33024): BF16_WIDE}.get((m, n), WIDE)
    if kind != "fp8":      # four K steps: below every line to the 128-tile kernel, and an even number
        name = {"bf16": "bf16", "fp4": "mxfp4"}[kind]
        assert routes.tile128_variant("fp8", m, n, 512) is None and not any(routes.rounds_on_128_tiles(m, n, 4, name, fp32=fp32) for fp32 in (False, True))
    check(kind, mode, m, n, k, kernel=kernel if kind == "fp8" else None)


# rows 4, 8, 16, 32 and 64 bytes past a multiple of 128 bytes, the first one too; bf16 rows on single elements
@pytest.mark.parametrize("c_pad,c_shift", [(2, 2), (4, 0), (1, 0), (0, 1), (8, 4), (16, 8), (32, 32), (64, 0)])
@pytest.mark.parametrize("m,n", [(2816, 4608), (2700, 4736)])
@pytest.mark.parametrize("kind,mode,k", [("fp8", g.TENSOR, 512), ("fp8", g.MX_TILED, 640), ("fp8", g.MX_TILED, 1536), ("fp8", g.MX_TILED, 1664)], ids=lambda v: str(v))
def test_rows_of_c_anywhere(c_pad, c_shift, m, n, kind, mode, k):
    check(kind, mode, m, n, k, c_pad=c_pad, c_shift=c_shift, kernel=BF16_WIDE if k == 640 else WIDE)


def test_batch_of_edges():
    check("fp8", g.ROWCOL, 2100, 2112, 512, batch=3, c_pad=2, c_shift=2, kernel=WIDE)
    check("fp8", g.MX_TILED, 2100, 2240, 768, batch=3, kernel=WIDE)
