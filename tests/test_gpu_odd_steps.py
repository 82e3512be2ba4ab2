"""An odd number of K steps (of 128 bytes) on the four-wave kernel, which walks them in pairs: the step behind the last one must add nothing,
whatever the bytes behind K hold; and row-major MX scales there, which it fetches 16 bytes of a row at a time.  Exact results (exact_gemm.py)."""
import pytest

import gcnasm_amd as g
import routes
from exact_gemm import check

# one round of ragged and of whole tiles, two tiles per workgroup, fp32 C past its own line; the fewest steps and more (the scale batches hold 8 or 4)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2790, 5111, 5), (2816, 5120, 7), (4090, 7100, 11), (2790, 5111, 13), (4350, 4200, 33)])
@pytest.mark.parametrize("kind", ["fp8", "fp4"])
def test_tiled_scales(m, n, steps, kind):
    # (bf16 C, fp32 C); the others run on the 128-tile kernel
    wide = {5: (True, False), 7: (True, False), 11: (True, kind == "fp8"), 13: (True, True), 33: (kind == "fp8", kind == "fp8")}[steps]
    assert tuple(routes.odd_tiled_mx_on_four_waves(m, n, steps, fp4=kind == "fp4", fp32=fp32) for fp32 in (False, True)) == wide
    check(kind, g.MX_TILED, m, n, steps * (256 if kind == "fp4" else 128))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp8", "fp4"])
def test_tiled_scales_of_a_batch(kind):
    assert routes.odd_tiled_mx_on_four_waves(2100, 2100, 5, batch=3)
    check(kind, g.MX_TILED, 2100, 2100, 5 * (256 if kind == "fp4" else 128), batch=3)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2790, 5111, 7), (2816, 5120, 13), (4090, 7100, 17)])
@pytest.mark.parametrize("pad", [0, 4, 8])                   # scale rows of 8 bytes a step: 8 (0), 12 (4) and 0 (8) bytes past a multiple of 16
def test_mxfp4_on_row_major_scales(m, n, steps, pad):
    assert routes.f4_row_scales_on_256_tiles(m, n, steps * 256)
    check("fp4", g.MX, m, n, steps * 256, pad=pad)


# scale rows of 4 bytes a step that start at every dword of a 16-byte piece (128, 132, 136, 140 bytes and four more); one round and two
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,steps", [(2300, 4099, 32), (2816, 5120, 33), (4350, 4200, 34), (4090, 7100, 33), (2300, 4099, 35)])
@pytest.mark.parametrize("pad", [0, 4])
def test_mxfp8_on_row_major_scales(m, n, steps, pad):
    assert routes.mx_row_scales_on_four_waves(steps)
    check("fp8", g.MX, m, n, steps * 128, pad=pad)


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [32, 33])
def test_mxfp8_on_row_major_scales_of_a_batch(steps):
    check("fp8", g.MX, 2100, 2100, steps * 128, batch=3, pad=4)


def test_rule_for_mxfp8_on_row_major_scales():
    for steps, wide in ((31, False), (32, True), (33, True)):
        assert routes.mx_row_scales_on_four_waves(steps) is wide
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, 4096, 4096, steps * 128, g.MX)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_persist")
        args.stride_sfa = (1 << 31) // 4096      # scale rows too far apart for 32-bit offsets past the end: still taken
        assert g.kernel_name(args) == "gemm_a8w8_persist"


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(2300, 4099), (4350, 4200)])
@pytest.mark.parametrize("kind,mode", [("fp8", g.ROWCOL), ("fp8", g.TENSOR), ("bf16", g.TENSOR)])
def test_scales_that_do_not_change_with_k(m, n, kind, mode):
    check(kind, mode, m, n, 33 * (64 if kind == "bf16" else 128))


@pytest.mark.parametrize("m,n,steps,fp4,fp32,wide", [
    (2816, 5120, 3, False, False, False), (2816, 5120, 5, False, False, True), (2816, 5120, 9, False, True, False), (2816, 5120, 11, False, True, True),
    (2816, 5120, 11, True, True, False), (2816, 5120, 13, True, True, True), (2304, 4096, 11, False, False, False), (2304, 4096, 13, False, False, True),
    (2304, 4096, 23, True, False, False), (2304, 4096, 25, True, False, True), (2304, 4096, 31, True, True, False), (2304, 4096, 33, True, True, True),
    (8192, 2560, 31, False, False, False), (8192, 2560, 33, False, True, True), (8192, 2560, 65, True, False, False)])
def test_rule_for_tiled_scales(m, n, steps, fp4, fp32, wide):
    assert routes.odd_tiled_mx_on_four_waves(m, n, steps, fp4=fp4, fp32=fp32) is wide
    if not fp4:
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, m, n, steps * 128, g.MX_TILED, g.FP32 if fp32 else g.BF16)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_tile128")
        if wide:      # C rows too far apart for 32-bit offsets: still taken, by the 128-tile kernel
            args.stride_c = 1 << 24
            assert g.kernel_name(args) == "gemm_a8w8_tile128"


def test_rule_for_scales_that_do_not_change_with_k():
    for steps, wide in ((31, False), (33, True)):
        assert routes.odd_steps_on_four_waves(steps) is wide
        args = g.raw_gemm_args(1 << 12, 1 << 12, 1 << 12, 1 << 12, 1 << 12, 4096, 4096, steps * 128, g.ROWCOL)
        assert g.kernel_name(args) == ("gemm_a8w8_wide" if wide else "gemm_a8w8_persist")
