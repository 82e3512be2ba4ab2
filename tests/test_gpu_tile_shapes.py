"""The tile shapes of the 128-tile kernel, each at sizes that take it: ragged edges in both directions, fewer K steps than LDS stages, as many and more,
every kind of operand and scale, shuffled weights, batches.  Exact results (exact_gemm.py)."""
import pytest

import gcnasm_amd as g
import routes
from exact_gemm import check

KINDS = [("fp8", g.ROWCOL, "fp8"), ("fp8", g.TENSOR, "fp8"), ("fp8", g.BLOCK, "block"), ("fp8", g.MX, "mx"), ("fp8", g.MX_TILED, "fp8"), ("bf16", g.TENSOR, "bf16"),
         ("fp4", g.MX, "mxfp4"), ("fp4", g.MX_TILED, "mxfp4_tiled")]
ELEMENTS = {"fp4": 256, "bf16": 64, "fp8": 128}               # of a K step


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps,batch,variant", [
    (129, 72, 2, 1, "64x64"), (200, 500, 3, 1, "64x64"), (321, 1000, 4, 1, "64x64"), (1024, 1024, 5, 1, "64x64"), (130, 250, 9, 5, "64x64"), (500, 700, 31, 1, "64x64"),
    (1000, 1400, 3, 1, "128x64"), (700, 1500, 8, 1, "128x64"), (600, 900, 15, 2, "128x64"), (1500, 1300, 28, 1, "128x64"), (1030, 1660, 33, 1, "128x64"),
    (2000, 1990, 2, 1, "128, four stages"), (1600, 2050, 5, 1, "128, four stages"), (700, 1700, 7, 2, "128, four stages")])
@pytest.mark.parametrize("kind,mode,route", KINDS, ids=lambda v: str(v))
def test_shapes(m, n, steps, batch, variant, kind, mode, route):
    if mode == g.BLOCK:
        n = (n + 127) // 128 * 128
    got = routes.tile128_variant(route, m, n, steps * 128, batch)
    assert got == variant or mode == g.BLOCK      # (whole blocks of columns are other sizes)
    check(kind, mode, m, n, steps * ELEMENTS[kind], batch=batch)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps,batch", [(200, 496, 3, 1), (321, 1008, 6, 1), (130, 256, 9, 5), (1000, 1408, 5, 1)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.MX_TILED), ("bf16", g.TENSOR), ("fp4", g.MX_TILED)], ids=lambda v: str(v))
def test_shuffled_weights(m, n, steps, batch, kind, mode):
    check(kind, mode, m, n, steps * ELEMENTS[kind], batch=batch, shuffled=True)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,variant", [(200, 500, 272, "64x64"), (321, 1000, 400, "64x64"), (140, 1300, 944, "64x64"), (1000, 1400, 624, "128x64"), (800, 2000, 2000, "128x64"),
                                           (1990, 2010, 336, "128, four stages")])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.TENSOR), ("bf16", g.TENSOR)], ids=lambda v: str(v))
def test_partial_steps(m, n, k, variant, kind, mode):
    assert routes.tile128_variant("block", m, n, k, 1) == variant or variant == "128, four stages"      # (no 256 x 128 tiles here either)
    check(kind, mode, m, n, k // 2 if kind == "bf16" else k)


def test_rule():
    for m, n, steps, kind, variant in ((129, 64, 1, "fp8", "64x64"), (1024, 1024, 64, "bf16", "64x64"), (1025, 1024, 64, "bf16", "128x64"), (1000, 1536, 8, "fp8", "128x64"),
                                       (256, 8192, 16, "mx", "128x64"), (256, 8192, 15, "mx", "128, four stages"), (2048, 2048, 8, "fp8", "128, four stages"),
                                       (2048, 2048, 8, "block", "128x64"), (1536, 1920, 8, "block", "128, four stages"), (128, 2048, 64, "fp8", "128x64"),
                                       (128, 2048, 8, "fp8", "128, four stages")):
        assert routes.tile128_variant(kind, m, n, steps * 128) == variant, (m, n, steps, kind)
