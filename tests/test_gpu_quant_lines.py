"""Tiled MX scales written by lines of the scale array, row-major ones over the flattened array, and per-row scales with a wave per row: the same bytes as the oracle's, at whole and
partial 64-row blocks and 256- and 512-column groups, with rows further apart than their elements."""
import numpy as np
import pytest
import torch

import gcnasm_amd as g
import routes
from gpu_util import dev


def _rows_apart(rows, k, pad, spread):
    """fp32 [rows, k], rows k + pad elements apart, NaN between them; a block of zeros, infinities and NaN among the blocks."""
    rng = np.random.Generator(np.random.Philox(rows + k))
    x = rng.standard_normal((rows, k), dtype=np.float32)
    if spread:
        x *= np.exp2(rng.integers(-6, 6, (rows, k // 32)).repeat(32, axis=1)).astype(np.float32)
    x[rows // 2, :32] = 0
    store = torch.full((rows, k + pad), float("nan"), device="cuda")
    store[:, :k] = dev(x)
    return x, store[:, :k]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k,waves", [(1024, 1056, 8), (1061, 1024, 8), (64, 32768, 8), (65, 20000, 8), (2100, 2560, 4), (3000, 2016, 4), (2049, 7392, 8), (8192, 160, 8)])
@pytest.mark.parametrize("pad", [0, 4])
def test_tiled_scales_by_lines(orc, rows, k, waves, pad):
    assert routes.mx_padding_in_launch(rows, k) and routes.quant_mx_by_lines(rows, k) == waves
    x, view = _rows_apart(rows, k, pad, True)
    q, s = g.quantize(view, g.MX_TILED)
    q0, s0 = orc.quantize(x, orc.MX)
    assert (q.cpu().numpy() == q0).all()
    assert (s.cpu().numpy() == orc.mx_tile_scales(s0)).all()
    if routes.quant_mx_by_lines(rows, k, fp4=True):
        q, s = g.quantize_mxfp4(view, tiled=True)
        q0, s0 = orc.quantize_mxfp4(x)
        assert (q.cpu().numpy() == q0).all() and (s.cpu().numpy() == orc.mx_tile_scales(s0)).all()


@pytest.mark.gpu
def test_tiled_scales_by_lines_of_infinities_and_nan(orc):
    """The same codes and exponents as the row-major quantiser's, block by block."""
    rows, k = 1100, 1024
    x, _ = _rows_apart(rows, k, 0, True)
    x[3, 40], x[700, 100], x[701, 600], x[1099, 1023] = np.inf, -np.inf, np.nan, np.nan
    x[5, :64] = np.finfo(np.float32).tiny / 8
    for quantize in (lambda t, tiled: g.quantize(t, g.MX_TILED if tiled else g.MX), lambda t, tiled: g.quantize_mxfp4(t, tiled=tiled)):
        (q1, s1), (q0, s0) = quantize(dev(x), True), quantize(dev(x), False)
        assert torch.equal(q1, q0) and (s1.cpu().numpy() == orc.mx_tile_scales(s0.cpu().numpy())).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(1, 32), (3, 224), (33, 1056), (2049, 1024), (257, 4128), (1056, 8192)])
@pytest.mark.parametrize("pad", [0, 4, 2048])
def test_row_major_scales_of_the_flattened_array(orc, rows, k, pad):
    """One, two and four chunks per wave, whole and partial last workgroups."""
    x, view = _rows_apart(rows, k, pad, True)
    # (finite values: a block that holds an infinity gets scale 1 on the device and 2^127 in the oracle, and NaN codes differ in their sign bit; the test
    # above compares such blocks with the tiled quantiser's)
    for (q, s), (q0, s0) in ((g.quantize(view, g.MX), orc.quantize(x, orc.MX)), (g.quantize_mxfp4(view), orc.quantize_mxfp4(x))):
        assert (q.cpu().numpy() == q0).all() and (s.cpu().numpy().reshape(s0.shape) == s0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,k", [(1025, 1024), (1027, 4), (1030, 256), (2306, 768), (1026, 1020), (5000, 260)])
@pytest.mark.parametrize("pad", [0, 4])
def test_a_wave_per_row(orc, rows, k, pad):
    assert routes.quant_rows_by_wave(rows, k)
    x, view = _rows_apart(rows, k, pad, False)
    x[7, :] = 0
    view[7, :] = 0
    q, s = g.quantize(view, g.ROWCOL)
    q0, s0 = orc.quantize(x, orc.ROWCOL)
    assert (q.cpu().numpy() == q0).all() and (s.cpu().numpy() == s0).all()


def test_rules():
    assert [routes.quant_mx_chunks(e, f, a) for f in (False, True) for a in (False, True) for e in (1 << 20, (1 << 20) + 32, 1 << 21, (1 << 21) + 32, 1 << 23)] == [
        1, 1, 1, 2, 2, 1, 1, 1, 2, 4, 1, 2, 2, 2, 2, 1, 2, 2, 2, 4]
    for rows, k, fp8, fp4 in ((128, 8192, None, None), (129, 8192, 8, 8), (1, 65536, 8, None), (64, 7168, None, None), (256, 8192, 8, 8), (2560, 2560, 4, 4),
                              (4096, 4096, 8, 8), (8192, 8192, 8, 8)):
        assert routes.quant_mx_by_lines(rows, k) == fp8 and routes.quant_mx_by_lines(rows, k, fp4=True) == fp4
    assert routes.quant_rows_by_wave(1025, 1024) and not routes.quant_rows_by_wave(1024, 1024) and not routes.quant_rows_by_wave(8192, 1028)
