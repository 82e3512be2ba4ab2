"""a8w8_quantize on the GPU against the oracle's quantisers: bytes and scales bit for bit (integer /
byte work), for every scale mode, ragged shapes, padded rows, all-zero groups and extreme magnitudes."""
import numpy as np
import pytest
import torch

import gcnasm_amd as g
import routes
from gpu_util import dev

pytestmark = pytest.mark.gpu


def _x(rows, k, seed, wide=True):
    rng = np.random.Generator(np.random.Philox(seed))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    if wide:
        x *= np.exp2(rng.integers(-30, 30, (rows, max(k // 32, 1)))).repeat(32, axis=1)[:, :k].astype(np.float32)
    x[rng.integers(0, rows), :] = 0            # an all-zero row
    return x


def _run(x, mode, group_rows=1):
    q, s = g.quantize(dev(x), mode, group_rows)
    torch.cuda.synchronize()
    return q.cpu().numpy(), s.cpu().numpy()


@pytest.mark.parametrize("rows,k", [(1, 32), (37, 96), (300, 1024), (2048, 4096)])
def test_per_tensor(orc, rows, k):
    x = _x(rows, k, 5 + rows, wide=False)
    q, s = _run(x, g.TENSOR)
    qr, sr = orc.quantize(x, orc.TENSOR)
    assert s.shape == (1,) and s.view(np.uint32)[0] == sr.view(np.uint32)[0]
    assert (q == qr).all()
    z = np.zeros((4, 64), np.float32)
    q, s = _run(z, g.TENSOR)
    assert s[0] == 1 and (q == 0).all()


@pytest.mark.parametrize("rows,k", [(1, 32), (37, 96), (256, 512), (130, 7168)])
def test_rowwise(orc, rows, k):
    x = _x(rows, k, 10 + rows)
    q, s = _run(x, g.ROWCOL)
    qr, sr = orc.quantize(x, orc.ROWCOL)
    assert (s.view(np.uint32) == sr.view(np.uint32)).all()
    assert (q == qr).all()


@pytest.mark.parametrize("rows,k", [(1, 128), (37, 384), (256, 2048)])
def test_block_1x128(orc, rows, k):
    x = _x(rows, k, 20 + rows)
    q, s = _run(x, g.BLOCK, 1)
    qr, sr = orc.quantize(x, orc.BLOCK, 1)
    assert s.shape == sr.shape and (s.view(np.uint32) == sr.view(np.uint32)).all()
    assert (q == qr).all()


@pytest.mark.parametrize("rows,k", [(128, 128), (384, 512)])
def test_block_128x128(orc, rows, k):
    x = _x(rows, k, 30 + rows)
    x[128:256, 0:128] = 0 if rows > 128 else x[128:256, 0:128]
    q, s = _run(x, g.BLOCK, 128)
    qr, sr = orc.quantize(x, orc.BLOCK, 128)
    assert s.shape == sr.shape and (s.view(np.uint32) == sr.view(np.uint32)).all()
    assert (q == qr).all()


@pytest.mark.parametrize("rows,k", [(1, 32), (37, 96), (256, 1024), (70, 7168)])
def test_mx(orc, rows, k):
    x = _x(rows, k, 40 + rows)
    x[0, :32] = [448 * 2.0 ** -3] + [0] * 31             # exactly a power of two times 448
    q, s = _run(x, g.MX)
    qr, sr = orc.quantize(x, orc.MX)
    assert (s == sr).all()
    assert (q == qr).all()


def test_extremes_and_padded_rows(orc):
    rows, k = 8, 256
    x = np.zeros((rows, k), np.float32)
    x[0, :4] = [3.0e38, -1.0e38, 1e-38, -1e-45]       # near fp32 max, a denormal
    x[1, :3] = [1e-40, 2e-40, -3e-41]                 # a row of denormals only
    x[2, :2] = [448.0, -447.9]
    x[3, 7] = -0.0
    for mode, gr in ((g.ROWCOL, 1), (g.BLOCK, 1), (g.MX, 1)):
        q, s = _run(x, mode, gr)
        qr, sr = orc.quantize(x, mode, gr)
        assert (q == qr).all(), mode
        assert (s.view(np.uint8) == sr.view(np.uint8)).all(), mode
    # a view with a row stride larger than k
    wide = _x(16, 512, 77)
    xv = dev(wide)[:, :256]
    q, s = g.quantize(xv, g.ROWCOL)
    qr, sr = orc.quantize(np.ascontiguousarray(wide[:, :256]), orc.ROWCOL)
    assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == sr).all()


def test_quantize_then_gemm_matches_oracle_pipeline(orc):
    """The bytes and scales a8w8_quantize writes feed a8w8_gemm directly, in every mode."""
    m, n, k = 256, 256, 512
    a, b = _x(m, k, 91, wide=False), _x(n, k, 92, wide=False)
    for mode, ga, gb in ((g.TENSOR, 1, 1), (g.ROWCOL, 1, 1), (g.BLOCK, 1, 128), (g.MX, 1, 1), (g.MX_TILED, 1, 1)):
        qa, sa = g.quantize(dev(a), mode, ga)
        qb, sb = g.quantize(dev(b), mode, gb)
        c = g.gemm(qa, qb, sa, sb, mode, c_dtype=g.FP32).cpu().numpy()
        omode = orc.MX if mode == g.MX_TILED else mode
        oa, osa = orc.quantize(a, omode, ga)
        ob, osb = orc.quantize(b, omode, gb)
        ref = orc.gemm_ref(oa, ob, osa, osb, omode)
        assert (np.abs(c - ref) <= 1e-2 * np.abs(ref) + 1e-2).all(), mode


def test_vector_and_scalar_kernels_agree_with_the_oracle_on_views(orc):
    """16-byte aligned rows take the vectorised kernels (four or eight elements per thread), anything
    else the one-element-per-thread kernels: an aligned view with padded rows, a view that starts four
    bytes into its rows, and a row longer than a workgroup holds in registers."""
    rows, k = 70, 512
    big = _x(rows, 2 * k + 32, 123)
    views = {"padded rows": (slice(None), slice(0, k)), "offset by one element": (slice(None), slice(1, 1 + k))}
    for name, (r, c) in views.items():
        want = np.ascontiguousarray(big[r, c])
        xv = dev(big)[r, c]
        assert (xv.data_ptr() % 16 == 0) == (name == "padded rows")
        for mode, gr in ((g.TENSOR, 1), (g.ROWCOL, 1), (g.BLOCK, 1), (g.MX, 1), (g.MX_TILED, 1)):
            q, s = g.quantize(xv, mode, gr)
            qr, sr = orc.quantize(want, orc.MX if mode == g.MX_TILED else mode, gr)
            assert (q.cpu().numpy() == qr).all(), (name, mode)
            if mode == g.MX_TILED:
                assert (s.cpu().numpy() == orc.mx_tile_scales(sr)).all(), (name, mode)
            else:
                assert (s.cpu().numpy().view(np.uint8) == sr.view(np.uint8)).all(), (name, mode)
        q4, s4 = g.quantize_mxfp4(xv)
        qr4, sr4 = orc.quantize_mxfp4(want)
        assert (q4.cpu().numpy() == qr4).all() and (s4.cpu().numpy() == sr4).all(), name
    long_rows = _x(5, 16384, 124)
    q, s = _run(long_rows, g.ROWCOL)
    qr, sr = orc.quantize(long_rows, orc.ROWCOL)
    assert (q == qr).all() and (s.view(np.uint32) == sr.view(np.uint32)).all()


@pytest.mark.parametrize("rows", [1, 7, 8, 9, 31, 33, 1025])
@pytest.mark.parametrize("k", [128, 2176])
def test_1x128_row_tiles(orc, rows, k):
    """Tiles of 8 rows (few blocks) and of 32 (1025 x 2176: more than 2^14 blocks), whole and ragged, and fewer than eight rows, which are
    taken along the rows; rows in a wider buffer."""
    x = np.random.default_rng(rows + k).standard_normal((rows, k)).astype(np.float32)
    x[0, :128] = 0
    whole = torch.full((rows, k + 4), 1e30, device="cuda")
    whole[:, :k] = dev(x)
    q, s = g.quantize(whole[:, :k], g.BLOCK)
    qr, sr = orc.quantize(x, orc.BLOCK, 1)
    assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == sr).all()
    if rows >= 128:
        x, whole = x[:1024], whole[:1024]
        q, s = g.quantize(whole[:, :k], g.BLOCK, 128)
        qr, sr = orc.quantize(x, orc.BLOCK, 128)
        assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == sr).all()


@pytest.mark.parametrize("rows,k", [(1, 32), (1, 4096), (63, 4096), (65, 992), (129, 2016), (300, 1024), (2049, 4096)])
def test_mx_quantisers_at_every_chunk_count(orc, rows, k):
    """Arrays of up to 2^18 elements, up to 2^23 and beyond (one, two and four chunks per wave; MXFP4 has two kernels), tiled
    layouts with padding rows and blocks; blocks whose largest value lies at, one ulp above and one ulp below a power of two times
    448 or 6, the smallest exponent with its subnormal quotients, Inf and NaN."""
    r = np.random.default_rng(rows + k)
    x = (r.standard_normal((rows, k)) * np.exp2(r.integers(-30, 30, (rows, k // 32)).repeat(32, axis=1))).astype(np.float32)
    for i, top in enumerate([448.0, 6.0]):
        for j, (e, ulp) in enumerate([(0, 0), (0, 1), (0, -1), (5, 1), (-127, 0), (-127, 1), (-127, 2), (-127, -1), (-128, 1)]):
            n = (2 * j + i) % (rows * (k // 32))
            v = np.float32(np.ldexp(top, e))
            block = x.reshape(-1, 32)[n]
            block[:] = 0
            block[7] = np.int32(v.view(np.int32) + ulp).view(np.float32)
    for mode, quantise, reference in [("e4m3", lambda t, tiled: g.quantize(t, g.MX_TILED if tiled else g.MX), lambda a: orc.quantize(a, orc.MX)),
                                      ("e2m1", lambda t, tiled: g.quantize_mxfp4(t, tiled=tiled), orc.quantize_mxfp4)]:
        qr, sr = reference(x)
        q, s = quantise(dev(x), False)
        assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == sr).all(), mode
        qt, st = quantise(dev(x), True)
        assert torch.equal(qt, q) and (st.cpu().numpy() == orc.mx_tile_scales(sr)).all(), mode


@pytest.mark.parametrize("rows,k", [(1, 4), (1, 4096), (3, 5460), (4, 4096), (1, 16388), (33, 516), (1024, 4096), (1025, 4100)])
def test_per_tensor_one_launch_and_three(orc, rows, k):
    """One workgroup up to 16384 elements, three launches beyond (one partial maximum, a few, all 1024 of them); the largest
    value in the last element and in the first, an all-zero array, NaN beside numbers."""
    for place in (0, rows * k - 1, None):
        x = np.random.default_rng(rows + k).standard_normal((rows, k)).astype(np.float32)
        if place is None:
            x[:] = 0
        else:
            x.reshape(-1)[place] = -77.5
            if rows * k > 8:
                x.reshape(-1)[rows * k // 2] = np.nan
        qr, sr = orc.quantize(np.nan_to_num(x, nan=0.0), orc.TENSOR)
        q, s = _run(x, g.TENSOR)
        number = ~np.isnan(x)
        assert s[0] == np.float32(sr).ravel()[0] and (q[number] == qr[number]).all()
        assert ((q[~number] & 0x7F) == 0x7F).all()


@pytest.mark.parametrize("k", [4, 4096, 4100, 8192, 8196, 16384, 16388])
def test_rowwise_at_every_row_length(orc, k):
    x = np.random.default_rng(k).standard_normal((5, k)).astype(np.float32)
    x[1] = 0
    x[2, k - 1] = 99.0
    qr, sr = orc.quantize(x, orc.ROWCOL)
    q, s = _run(x, g.ROWCOL)
    assert (q == qr).all() and (s == sr).all()


def test_per_tensor_beyond_the_threads_of_one_launch():
    """2^35 elements, 128 GiB of them: one thread per eight elements would be 2^32 threads, more than a launch takes."""
    rows, k = 1 << 20, 1 << 15
    if torch.cuda.mem_get_info()[0] < 180 << 30:
        pytest.skip("needs 160 GiB of free memory")
    x = torch.empty((rows, k), device="cuda")
    x.uniform_(-1.0, 1.0)
    x[rows - 1, k - 3] = -896.0
    q, s = g.quantize(x, g.TENSOR)
    assert float(s) == 2.0
    for first in (0, 1, rows // 2, rows - 3):
        want = g.cvt_f32_to_e4m3(x[first:first + 3] / 2.0)
        assert torch.equal(q[first:first + 3], want), first
    del x, q
    torch.cuda.empty_cache()


@pytest.mark.parametrize("rows,k", [(1, 131072), (3, 140000 // 32 * 32), (16384, 32), (16385, 96), (9000, 544)])
def test_tiled_scales_with_much_padding(orc, rows, k):
    """More than three million padding elements: their scales come from a fill launch, the others from a quantiser over the real ones."""
    assert not routes.mx_padding_in_launch(rows, k)
    x = np.random.default_rng(rows + k).standard_normal((rows, k)).astype(np.float32)
    for q, s, qr, sr in [(*g.quantize(dev(x), g.MX_TILED), *orc.quantize(x, orc.MX)), (*g.quantize_mxfp4(dev(x), tiled=True), *orc.quantize_mxfp4(x))]:
        assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == orc.mx_tile_scales(sr)).all()


@pytest.mark.parametrize("rows,k", [(1, 128), (1, 1152), (2, 128), (3, 1152), (5, 70016), (7, 1152), (8, 1152), (9, 1 << 19), (31, 70016), (33, (1 << 19) + 128)])
def test_1x128_few_rows(orc, rows, k):
    """Along the rows (fewer than eight of them, or long ones), eight rows per workgroup, and the lines between; an all-zero group, a
    padded input."""
    assert routes.quant_1x128_along_rows(rows, k) is (rows < 8 or k >= 1 << 19)
    x = np.random.default_rng(rows * k).standard_normal((rows, k)).astype(np.float32)
    x[rows - 1, k - 128:] = 0
    whole = torch.full((rows, k + 8), 1e30, device="cuda")
    whole[:, :k] = dev(x)
    q, s = g.quantize(whole[:, :k], g.BLOCK)
    qr, sr = orc.quantize(x, orc.BLOCK, 1)
    assert (q.cpu().numpy() == qr).all() and (s.cpu().numpy() == sr).all()
