"""The order of tiles over the XCDs, a run each or every eighth tile, on counts that 8 does not divide: every tile of C is computed, in every kernel that has the
choice.  Exact results (exact_gemm.py)."""
import pytest

import gcnasm_amd as g
import routes
from exact_gemm import check


# 64 x 64, 128 x 64, 128 x 128 and 256 x 128 tiles; the last group of rows full but for one, and one row
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps,batch,bm,bn,runs", [
    (200, 900, 3, 1, 64, 64, True), (440, 380, 3, 5, 64, 64, True), (580, 900, 3, 1, 64, 64, False), (1080, 700, 3, 1, 64, 64, False), (580, 400, 2, 3, 64, 64, False),
    (600, 1088, 40, 1, 64, 64, True), (700, 1900, 3, 1, 128, 64, True), (200, 350, 17, 16, 128, 64, False), (900, 880, 30, 8, 256, 128, False), (2200, 700, 16, 1, 128, 64, False),
    (600, 4300, 3, 1, 128, 128, True), (2200, 1700, 3, 1, 128, 128, False), (1153, 3700, 3, 1, 128, 128, True), (2177, 2600, 3, 1, 128, 128, False),
    (700, 6700, 24, 1, 256, 128, True), (3300, 2300, 24, 1, 256, 128, False)])
@pytest.mark.parametrize("kind,mode,route", [("fp8", g.ROWCOL, "fp8"), ("bf16", g.TENSOR, "bf16")], ids=lambda v: str(v))
def test_128_tiles(m, n, steps, batch, bm, bn, runs, kind, mode, route):
    variant = routes.tile128_variant(route, m, n, steps * 128, batch)
    assert variant == {(64, 64): "64x64", (128, 64): "128x64", (256, 128): "256x128"}.get((bm, bn), variant)
    tiles = -(-m // bm), -(-n // bn)
    assert tiles[0] * tiles[1] % 8 and routes.tiles_in_runs(*tiles, steps, batch, bm > bn) is runs
    check(kind, mode, m, n, steps * (64 if kind == "bf16" else 128), batch=batch)


# four waves, eight waves, 128-tiles in badly filled rounds
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps,batch,runs", [(2100, 5200, 4, 1, False), (2100, 5200, 26, 1, True), (1500, 5700, 4, 1, True), (2600, 3300, 4, 3, False), (5300, 7300, 4, 1, True)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.MX_TILED), ("fp8", g.BLOCK), ("fp8", g.MX)], ids=lambda v: str(v))
def test_256_tiles(m, n, steps, batch, runs, kind, mode):
    n = (n + 127) // 128 * 128 if mode == g.BLOCK else n
    tiles = -(-m // 256), -(-n // 256)
    assert tiles[0] * tiles[1] % 8 and routes.items_in_runs(*tiles, steps, batch) is runs
    name = "gemm_a8w8_wide" if mode in (g.ROWCOL, g.MX_TILED) else "gemm_a8w8_persist"
    check(kind, mode, m, n, steps * 128, batch=batch, kernel={g.BF16: name, g.FP32: name})


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,runs", [(6300, 2900, True), (4300, 4750, True), (7300, 1600, False)])
def test_128_tiles_in_rounds(m, n, runs):
    tiles = -(-m // 128), -(-n // 128)
    assert tiles[0] * tiles[1] % 8 and routes.tiles_in_runs(*tiles, 5) is runs and routes.rounds_on_128_tiles(m, n, 5)
    check("fp8", g.ROWCOL, m, n, 640, kernel={g.BF16: "gemm_a8w8_tile128", g.FP32: "gemm_a8w8_tile128"})


def test_rules():
    assert all(routes.tiles_in_runs(a, b, 1) and routes.items_in_runs(a, b, 1) for a, b in ((8, 7), (16, 5), (100, 4), (9, 8)))
    for tiles, steps, batch, tall, runs in (((7, 3), 9, 1, False, True), ((7, 3), 9, 8, False, True), ((2, 6), 9, 16, True, False), ((2, 6), 9, 16, False, True), ((2, 6), 9, 1, True, True), ((4, 7), 50, 8, True, False), ((4, 7), 50, 8, False, True),
                                            ((3, 6), 9, 16, True, True), ((9, 9), 9, 1, False, False), ((9, 28), 39, 1, False, False), ((9, 28), 40, 1, False, True),
                                            ((17, 12), 50, 1, False, False), ((9, 29), 9, 1, False, True), ((17, 17), 9, 1, False, False), ((25, 21), 9, 1, False, True),
                                            ((59, 13), 9, 1, False, False)):
        assert routes.tiles_in_runs(*tiles, steps, batch, tall) is runs, (tiles, steps, batch, tall)
    for tiles, steps, batch, runs in (((7, 29), 2, 1, True), ((9, 28), 15, 1, False), ((9, 28), 16, 1, True), ((9, 9), 4, 6, False), ((9, 9), 4, 7, True), ((31, 31), 4, 1, True)):
        assert routes.items_in_runs(*tiles, steps, batch) is runs, (tiles, steps, batch)
