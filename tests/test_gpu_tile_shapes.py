"""The tile shapes of the 128-tile kernel, each at sizes that take it: ragged edges in both directions, fewer K steps than LDS stages, as many and more,
every kind of operand and scale, shuffled weights, batches.  Exact results (exact_gemm.py)."""
import ctypes

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
    want = {g.BF16: variant, g.FP32: variant}
    if mode == g.BLOCK:      # whole blocks of columns are other sizes, and fp32 C has a line of its own
        want.update({(1500, 1408): {g.BF16: "128, four stages", g.FP32: "128, four stages"}, (2000, 2048): {g.FP32: "128x64"}, (1600, 2176): {g.FP32: "128x64"}}.get((m, n), {}))
    assert {c: routes.tile128_variant(route, m, n, steps * 128, batch, fp32=c == g.FP32) for c in want} == want
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
    assert routes.tile128_variant("fp8", m, n, k, 1) == variant
    check(kind, mode, m, n, k // 2 if kind == "bf16" else k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(3080, 5120, 5), (4352, 4608, 6), (5300, 4096, 8)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.BLOCK), ("fp8", g.MX), ("fp8", g.MX_TILED), ("bf16", g.TENSOR), ("fp4", g.MX_TILED)], ids=lambda v: str(v))
def test_shuffled_weights_in_badly_filled_rounds(m, n, steps, kind, mode):
    check(kind, mode, m, n, steps * ELEMENTS[kind], shuffled=True)


# more than two 128-tiles per compute unit, in rounds that 256-tiles fill badly
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(4352, 4608, 5), (6100, 3001, 6), (2100, 4200, 8), (5300, 4000, 16)])
@pytest.mark.parametrize("kind,mode,route", [k for k in KINDS if k != ("fp4", g.MX, "mxfp4")], ids=lambda v: str(v))
def test_badly_filled_rounds(m, n, steps, kind, mode, route):
    n = n // 128 * 128 if mode == g.BLOCK else n
    name = {"fp8": {g.MX_TILED: "mxfp8", g.MX: "mx", g.BLOCK: "block"}.get(mode, "fp8"), "fp4": "mxfp4"}.get(kind, kind)
    # (bf16 C, fp32 C); the others run on 256-tiles
    small = {8: {"mxfp8": (False, True), "mx": (False, True), "block": (False, True)}, 16: {"mxfp8": (False, False), "mx": (False, False), "mxfp4": (False, True)}}.get(steps, {})
    assert routes.tile128_variant(route, m, n, steps * 128) is None
    assert tuple(routes.rounds_on_128_tiles(m, n, steps, name, fp32=fp32) for fp32 in (False, True)) == small.get(name, (True, True))
    check(kind, mode, m, n, steps * ELEMENTS[kind])


def test_rule_for_badly_filled_rounds():
    for m, n, steps, kind, fp32, small in ((4352, 4608, 4, "fp8", False, False), (4352, 4608, 5, "fp8", False, True), (4352, 4608, 32, "bf16", True, True), (4352, 4608, 33, "fp8", True, False),
                                           (4352, 4608, 20, "mxfp8", False, True), (4352, 4608, 22, "mxfp8", False, False), (4352, 4608, 32, "mxfp4", False, True),
                                           (2304, 4096, 16, "fp8", False, True), (2304, 4096, 18, "fp8", False, False), (2304, 4096, 6, "mxfp8", False, False), (2304, 4096, 8, "mxfp8", True, True),
                                           (2304, 4096, 10, "mxfp4", False, False), (2304, 4096, 16, "mxfp4", True, True), (4096, 4096, 8, "fp8", False, False),
                                           (4096, 7168, 8, "fp8", False, False), (8192, 4608, 8, "fp8", False, False), (4352, 4608, 32, "block", False, True),
                                           (5376, 4096, 24, "block", False, True), (5376, 4096, 26, "block", True, False), (2304, 4096, 8, "block", False, False),
                                           (2304, 4096, 16, "block", True, True), (4352, 4608, 16, "mx", False, True), (4352, 4608, 18, "mx", True, False),
                                           (5376, 4096, 8, "mx", False, True), (5376, 4096, 10, "mx", False, False), (2304, 4096, 12, "mx", True, True)):
        assert routes.rounds_on_128_tiles(m, n, steps, kind, fp32=fp32) is small, (m, n, steps, kind, fp32)
        if kind in ("fp8", "mxfp8", "block", "mx"):
            args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, steps * 128, {"fp8": g.ROWCOL, "mxfp8": g.MX_TILED, "block": g.BLOCK, "mx": g.MX}[kind], g.FP32 if fp32 else g.BF16)
            assert (g.kernel_name(args) == "gemm_a8w8_tile128") is small
            args.stride_c = 1 << 24          # past the 256-tile kernels' offsets: refused, as before
            if steps % 2 == 0:
                assert g.kernel_name(args) in ("gemm_a8w8_wide", "gemm_a8w8_persist") and g.lib().a8w8_gemm(ctypes.byref(args), None) == -7


@pytest.mark.parametrize("m,n,batch,most", [(953, 640, 16, 8), (700, 768, 16, 8), (1020, 1280, 8, 10), (2600, 2176, 2, 16), (2304, 4096, 1, 16)])
def test_rounds_of_a_batch_of_small_entries(m, n, batch, most):
    """Three rounds of 128-tiles against one of 256-tiles, up to `most` steps: beyond, small entries took up to 1.26 times as long."""
    for kind, fp32 in (("bf16", False), ("bf16", True), ("fp8", False), ("block", True)):
        assert [routes.rounds_on_128_tiles(m, n, s, kind, batch, fp32) for s in (5, most, most + 1)] == [True, True, False], (kind, fp32)


def test_rounds_over_shuffled_weights():
    """Measured on row-major weights, the rounds made shuffled ones up to 1.25 times as slow."""
    four, five, six, three = (3080, 5120), (4352, 4608), (5376, 4096), (2304, 4096)      # rounds of 128-tiles, against 2, 2, 2 and 1 of 256-tiles
    for kind, bf16_most, fp32_most in (("fp8", 0, 12), ("bf16", 0, 12), ("block", 0, 16), ("mx", 0, 8), ("mxfp8", 20, 20), ("mxfp4", 32, 32)):
        for fp32, most in ((False, bf16_most), (True, fp32_most)):
            assert [routes.rounds_on_128_tiles(*five, s, kind, fp32=fp32, shuffled=True) for s in (5, most, most + 1)] == [most > 0, most > 0, False], (kind, fp32)
            assert not routes.rounds_on_128_tiles(*six, 5, kind, fp32=fp32, shuffled=True) and not routes.rounds_on_128_tiles(*three, 5, kind, fp32=fp32, shuffled=True)
            assert routes.rounds_on_128_tiles(*four, 8, kind, fp32=fp32, shuffled=True) and routes.rounds_on_128_tiles(*four, 8, kind, fp32=fp32)
    for mode, shuffled, name in ((g.ROWCOL, 0, "gemm_a8w8_tile128"), (g.ROWCOL, 1, "gemm_a8w8_wide"), (g.BLOCK, 0, "gemm_a8w8_tile128"), (g.BLOCK, 1, "gemm_a8w8_persist")):
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, *six, 1024, mode, b_preshuffled=shuffled)
        assert g.kernel_name(args) == name


def test_rule():
    for m, n, steps, kind, variant in ((129, 64, 1, "fp8", "64x64"), (1024, 1024, 64, "bf16", "64x64"), (1025, 1024, 64, "bf16", "128x64"), (1000, 1536, 8, "fp8", "128x64"),
                                       (256, 8192, 16, "mx", "128x64"), (256, 8192, 15, "mx", "128, four stages"), (2048, 2048, 8, "fp8", "128, four stages"),
                                       (2048, 2048, 8, "block", "128x64"), (1536, 1920, 8, "block", "128, four stages"), (128, 2048, 64, "fp8", "128x64"),
                                       (128, 2048, 8, "fp8", "128, four stages")):
        assert routes.tile128_variant(kind, m, n, steps * 128) == variant, (m, n, steps, kind)


@pytest.mark.parametrize("m,n,batch", [(24640, 128, 1), (3200, 1024, 1), (1600, 2048, 1), (2300, 1536, 1), (4500, 896, 1), (2048, 2048, 1), (512, 512, 16), (976, 512, 8), (512, 1024, 7)])
@pytest.mark.parametrize("steps", [3, 8, 9, 32])
def test_block_scales_up_to_one_tile_per_compute_unit(m, n, batch, steps):
    """193 to 256 tiles of 128 x 128 are halved for fp32 C, few steps and eight columns of them only: elsewhere two halves on a compute unit take up to 1.5 times as long."""
    assert 192 < batch * -(-m // 128) * (n // 128) <= 256
    assert routes.tile128_variant("block", m, n, steps * 128, batch, fp32=False) == "128, four stages"
    assert routes.tile128_variant("block", m, n, steps * 128, batch, fp32=True) == ("128x64" if steps <= 8 and n >= 1024 else "128, four stages")


def test_stages_of_128x64_tiles():
    """Up to 128 rows the weights come from HBM: deep staging for every kind of step."""
    for kind in ("fp8", "bf16", "mxfp8", "block", "mx", "mxfp4", "mxfp4_tiled", "ragged"):
        light = kind in ("fp8", "bf16", "mxfp8")
        assert [routes.narrow_tiles_deep(kind, m, s * 128) for m, s in ((1, 16), (128, 16), (128, 64), (129, 27), (129, 28))] == [True, True, True, False, light]


def test_stages_of_128x64_tiles_over_large_weights():
    """Up to 384 rows too, light steps from 12 MiB of weights and block scales from 20: three stages took up to 13% longer from HBM."""
    for kind, mib in (("fp8", 12), ("bf16", 12), ("mxfp8", 12), ("block", 20)):
        assert [routes.narrow_tiles_deep(kind, m, 2048, n) for m, n in ((129, mib * 512), (384, mib * 512), (385, mib * 512), (384, mib * 512 - 1))] == [True, True, False, False]
    assert not any(routes.narrow_tiles_deep(kind, 129, 8192, 8192) for kind in ("mx", "mxfp4", "mxfp4_tiled", "ragged"))


# deep staging up to 128 rows: fewer, as many and more K steps than twice the stages; the last one a partial step
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(1, 200, 16), (100, 1000, 17), (128, 1990, 30)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.MX), ("fp4", g.MX), ("fp8", g.BLOCK)], ids=lambda v: str(v))
def test_up_to_128_rows(m, n, steps, kind, mode):
    n = (n + 127) // 128 * 128 if mode == g.BLOCK else n
    assert routes.tile128_variant("block", m, n, steps * 128) == "128x64"
    check(kind, mode, m, n, steps * ELEMENTS[kind])


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps,kind,mode", [(200, 6400, 26, "block", g.BLOCK), (300, 4992, 33, "block", g.BLOCK), (190, 6500, 16, "fp8", g.ROWCOL), (257, 5300, 19, "fp8", g.MX_TILED),
                                                 (130, 7000, 27, "bf16", g.TENSOR)])
def test_deep_staging_over_large_weights(m, n, steps, kind, mode):
    assert routes.tile128_variant("fp8", m, n, steps * 128) == "128x64" and routes.narrow_tiles_deep({"fp8": "mxfp8"}.get(kind, kind), m, steps * 128, n)
    check("fp8" if kind == "block" else kind, mode, m, n, steps * (64 if kind == "bf16" else 128))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 200, 2064), (100, 1000, 2032), (128, 1990, 4016)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.TENSOR), ("bf16", g.TENSOR)], ids=lambda v: str(v))
def test_up_to_128_rows_partial_steps(m, n, k, kind, mode):
    assert routes.tile128_variant("fp8", m, n, k) == ("128, four stages" if k == 2032 else "128x64")      # (2032: a step short of narrow tiles)
    check(kind, mode, m, n, k // 2 if kind == "bf16" else k)
