"""The size rules of the dispatch, at sizes where the variants on their two sides were measured to differ."""
import pytest

import gcnasm_amd as g
import routes


@pytest.mark.parametrize("rows,k,in_launch", [(1, 4096, True), (16, 7168, True), (1, 65536, True), (4096, 32, True), (8192, 8320, True), (16384, 288, False),
                                              (1, 131072, False), (16, 262144, False), (1, 1 << 20, False), (16384, 32, False),
                                              (65536, 32, False), (262144, 96, False), (65536, 1056, False),
                                              (64, 1 << 20, True), (1 << 20, 2048, False), ((1 << 20) - 1, 2048, False)])
def test_padding_of_tiled_mx_scales(rows, k, in_launch):
    """Padded in the quantiser's own launch up to four million elements in all or three million of padding; arrays without padding always (the grid is the same)
    as long as their elements can be counted with 31 bits."""
    assert routes.mx_padding_in_launch(rows, k) is in_launch


@pytest.mark.parametrize("m,n,k,tiles", [(128, 260, 16, False), (128, 512, 16, False), (129, 1000, 16, False), (256, 1024, 16, True), (64, 260, 48, False),
                                         (128, 260, 48, False), (128, 512, 32, True), (64, 260, 80, True), (37, 53, 96, False), (46, 46, 240, False),
                                         (300, 391, 240, True), (1, 16, 272, True), (1000, 3000, 2000, True)])
def test_partial_k_steps(m, n, k, tiles):
    """On the tiles from 256 bytes of K on, below by the multiply-adds: the library's own choice, too."""
    assert routes.partial_steps_on_tiles(m, n, k) is tiles
    args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, k, g.ROWCOL)
    assert g.kernel_name(args) == ("gemm_a8w8_tile128" if tiles else "gemm_a8w8_general")


@pytest.mark.parametrize("n,few", [(1, True), (65536, True), ((1 << 20) + 3, True), ((1 << 21) - 1, True), (1 << 21, False), (1 << 25, False), (1 << 40, False)])
def test_fnuz_conversions(n, few):
    assert routes.cvt_fnuz_few(n) is few


@pytest.mark.parametrize("rows,k,along", [(1, 128, True), (1, 1 << 20, True), (3, 1 << 20, True), (7, 4096, True), (8, 4096, False), (17, 1 << 20, True),
                                          (65, 1 << 20, True), (65, 65536, False), (128, 1 << 20, False), (8192, 8192, False)])
def test_1x128_quantiser(rows, k, along):
    assert routes.quant_1x128_along_rows(rows, k) is along


@pytest.mark.parametrize("m,n,k,bf16,fp32", [(4096, 4096, 512, False, False), (4096, 4096, 1024, True, False), (4096, 4096, 2048, True, True),
                                             (8192, 8192, 8192, True, True), (4096, 7168, 1024, True, False), (4096, 7168, 3072, True, True),
                                             (3000, 8192, 2048, False, False), (3000, 8192, 3072, True, False), (3000, 8192, 4096, True, True),
                                             (8192, 2560, 512, False, False), (8192, 2560, 8192, False, False), (4096, 2560, 2048, False, False),
                                             (4096, 2560, 4096, True, True)])
def test_mxfp4_row_major_scales_past_two_tiles_per_compute_unit(m, n, k, bf16, fp32):
    assert routes.f4_row_scales_on_256_tiles(m, n, k) is bf16
    assert routes.f4_row_scales_on_256_tiles(m, n, k, fp32=True) is fp32


# the flat GEMM's splits on both sides of their lines, 256 compute units; (weight tiles, row groups) per workgroup
@pytest.mark.parametrize("kind,row_major,m,n,k,split", [
    ("fp8", False, 16, 4096, 4096, (1, 1)), ("fp8", False, 16, 5120, 8192, (2, 1)), ("fp8", True, 16, 5120, 8192, (2, 1)),
    ("fp8", True, 1, 7168, 8192, (1, 1)), ("bf16", True, 4, 6144, 4096, (1, 1)), ("bf16", True, 4, 6144, 8192, (2, 1)), ("block", True, 1, 7168, 8192, (2, 1)),
    ("mxfp8", True, 1, 7168, 8192, (2, 1)), ("fp8", False, 16, 10240, 8192, (4, 1)), ("fp8", False, 16, 10240, 1024, (4, 1)), ("fp8", False, 8, 10240, 1024, (2, 1)), ("fp8", False, 16, 14336, 1024, (2, 1)),
    ("fp8", True, 16, 9216, 512, (2, 1)), ("fp8", False, 1, 14336, 8192, (2, 1)), ("fp8", False, 16, 14336, 8192, (4, 1)),
    ("bf16", False, 8, 15360, 4096, (2, 1)), ("fp8", True, 1, 12288, 2048, (2, 1)), ("fp8", True, 8, 13312, 8192, (4, 1)), ("mxfp8", True, 1, 14336, 2048, (2, 1)),
    ("mxfp8", True, 16, 14336, 2048, (4, 1)), ("fp8", False, 32, 14336, 1024, (2, 2)), ("fp8", False, 32, 14336, 4096, (4, 2)),
    ("block", False, 48, 14336, 1024, (2, 3)), ("block", False, 64, 14336, 1024, (4, 4)), ("fp8", True, 64, 14336, 512, (4, 4)), ("fp8", False, 64, 14336, 512, (2, 4)),
    ("mxfp4", False, 64, 12288, 1024, (2, 4)), ("mxfp4", False, 64, 12288, 4096, (4, 4)), ("mxfp8", False, 48, 14336, 1024, (4, 3)), ("fp8", False, 96, 8192, 8192, (2, 6)),
    ("mxfp8", False, 96, 8192, 8192, (4, 4)), ("mxfp4", False, 80, 5120, 1024, (2, 6)), ("fp8", False, 128, 8192, 8192, (4, 4)), ("fp8", False, 128, 12288, 2560, (2, 4)),
    ("fp8", False, 100, 1024, 4096, (1, 2)), ("fp8", False, 48, 16384, 7168, (4, 3)), ("fp8", False, 80, 16384, 7168, (4, 3)), ("fp8", False, 128, 16384, 7168, (4, 4))])
def test_flat_splits(kind, row_major, m, n, k, split):
    assert routes.flat_split(kind, row_major, m, n, k) == split


@pytest.mark.parametrize("kind,row_major,m,n,k,batch,flat", [
    ("fp8", False, 16, 16384, 7168, 1, True), ("fp8", False, 128, 16384, 7168, 1, False), ("fp8", False, 128, 8192, 8192, 1, True),
    ("mxfp8", True, 128, 8192, 8192, 4, False), ("mxfp8", True, 128, 8192, 8192, 2, False), ("bf16", False, 96, 8192, 8192, 2, False),
    ("fp8", True, 64, 14336, 14336, 2, False), ("fp8", True, 64, 14336, 4096, 2, True), ("mxfp4", True, 64, 14336, 14336, 4, False),
    ("block", False, 64, 14336, 4096, 4, False), ("fp8", True, 64, 8192, 8192, 4, True), ("bf16", True, 64, 8192, 8192, 4, True),
    ("fp8", False, 96, 4096, 4096, 16, True)])
def test_flat_against_dense(kind, row_major, m, n, k, batch, flat):
    """The side of cells whose two sides were measured to be more than 5% apart; a batch counts where more than four row groups share
    the weights of an entry, and past 128 MiB of weights between two and four weight tiles per compute unit."""
    assert routes.flat_is_faster(kind, row_major, m, n, k, batch) is flat
    if kind in ("fp8", "mxfp8", "block"):
        mode = {"fp8": g.ROWCOL, "mxfp8": g.MX_TILED, "block": g.BLOCK}[kind]
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, k, mode, batch=batch, b_preshuffled=int(not row_major))
        assert (g.kernel_name(args) == "flatmm_a8w8") is flat


@pytest.mark.parametrize("kind,m,n,k_bytes,batch,variant", [
    ("fp8", 256, 8192, 8192, 1, "128x64"), ("fp8", 256, 8192, 1920, 1, "128, four stages"), ("fp8", 2048, 2048, 2048, 1, "128, four stages"),
    ("fp8", 2560, 2560, 2560, 1, "256x128"), ("fp8", 2560, 2560, 1920, 1, "128, two stages"), ("block", 2560, 2560, 2560, 1, "128, two stages"),
    ("bf16", 2560, 2560, 3072, 1, "256x128"), ("bf16", 2560, 2560, 2944, 1, "128, two stages"), ("mxfp4_tiled", 2560, 2560, 2048, 1, "128, two stages"),
    ("mxfp4", 2560, 2560, 2048, 1, "256x128"), ("fp8", 512, 16384, 7168, 1, "256x128"), ("fp8", 129, 16400, 2048, 1, "256x128"),
    ("fp8", 129, 16400, 2048, 2, None), ("fp8", 4096, 4096, 4096, 1, None)])
def test_128_tile_kernel(kind, m, n, k_bytes, batch, variant):
    assert routes.tile128_variant(kind, m, n, k_bytes, batch) == variant
