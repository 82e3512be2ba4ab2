"""How the flat GEMM deals weight tiles and row groups to workgroups, against exact products, on pre-shuffled and on row-major weights:
layers from a few weight tiles to more than two per compute unit with two to eight groups of 16 rows, ragged last ones (test_fp8,
test_mxfp4_and_bf16), and every split that its rule can choose, for every kind of operands (test_every_split_is_exact)."""
import pytest
import torch

import gcnasm_amd as g
import routes

pytestmark = pytest.mark.gpu


def _scaled(gen, rows, k, mode, weight):
    x = torch.randint(-4, 5, (rows, k), generator=gen, device="cuda").float()
    codes = g.cvt_f32_to_e4m3(x)
    two = lambda *shape: torch.exp2(torch.randint(-2, 3, shape, generator=gen, device="cuda").float())
    if mode in (g.TENSOR, g.ROWCOL):
        s = two(rows if mode == g.ROWCOL else 1)
        return codes, s, x.double() * s[:, None]
    if mode == g.BLOCK:
        s = two(rows // 128, k // 128) if weight else two(k // 128, rows)
        full = s.repeat_interleave(128, 0).repeat_interleave(128, 1) if weight else s.T.repeat_interleave(128, 1)
        return codes, s, x.double() * full
    e = torch.randint(125, 130, (rows, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
    return codes, g.mx_tile_scales(e), x.double() * torch.exp2(e.double() - 127).repeat_interleave(32, 1)


@pytest.mark.parametrize("mode", [g.TENSOR, g.ROWCOL, g.BLOCK, g.MX_TILED])
@pytest.mark.parametrize("n", [1024, 2176, 4096, 8192, 9216])
def test_fp8(n, mode):
    gen = torch.Generator(device="cuda").manual_seed(n + mode)
    k = 512 + 128
    b, sb, B = _scaled(gen, n, k, mode, True)
    shuffled = g.preshuffle_b_device(b)
    for m in (17, 40, 64, 65, 96, 101, 128):
        a, sa, A = _scaled(gen, m, k, mode, False)
        ref = (A @ B.T).float()
        for c_dtype, want in ((g.FP32, ref), (g.BF16, ref.bfloat16())):
            assert torch.equal(g.flatmm(a, shuffled, sa, sb, n, scale_mode=mode, c_dtype=c_dtype), want), (m, n)
            assert torch.equal(g.gemm(a, b, sa, sb, mode, c_dtype=c_dtype), want), (m, n, "row-major")


@pytest.mark.parametrize("n", [1040, 4096, 8192, 9232])
def test_mxfp4_and_bf16(n):
    gen = torch.Generator(device="cuda").manual_seed(n)
    k = 768
    value = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
    value = torch.cat([value, -value])

    def operand(rows):
        c = torch.randint(0, 16, (rows, k), generator=gen, device="cuda")
        e = torch.randint(125, 130, (rows, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        q = (c[:, ::2] | c[:, 1::2] << 4).to(torch.uint8)
        return q, g.mx_tile_scales(e), value[c] * torch.exp2(e.double() - 127).repeat_interleave(32, 1)

    qb, sb, B = operand(n)
    b16 = torch.randint(-4, 5, (n, k), generator=gen, device="cuda").bfloat16()
    shuffled, shuffled16 = g.preshuffle_b_device(qb), g.preshuffle_b_bf16_device(b16)
    for m in (17, 48, 64, 80, 113, 128):
        qa, sa, A = operand(m)
        ref = (A @ B.T).float()
        assert torch.equal(g.flatmm_a4w4(qa, shuffled, sa, sb, n, c_dtype=g.FP32), ref), (m, n)
        assert torch.equal(g.gemm_a4w4(qa, qb, sa, sb, c_dtype=g.FP32), ref), (m, n, "row-major")
        a16 = torch.randint(-4, 5, (m, k), generator=gen, device="cuda").bfloat16()
        ref = (a16.double() @ b16.double().T).float()
        assert torch.equal(g.flatmm_a16w16(a16, shuffled16, n, c_dtype=g.FP32), ref), (m, n, "bf16")
        assert torch.equal(g.gemm_a16w16(a16, b16, c_dtype=g.FP32), ref), (m, n, "bf16 row-major")


# Every split of every kind of operands in both layouts: (weight tiles, row groups) per workgroup, M, N, K.  Odd counts of weight tiles
# (the last workgroup of two or four is not full) where N need not be whole 128-wide blocks.
def _split_cases(kind, row_major):
    odd, two = (4224, 8320) if kind == "block" else (4112, 8208)
    few, short, long = (1024 if kind == "block" else 1008), 512, (2560 if kind != "mxfp4" else 5120)
    cases = [((1, 1), 16, few, 640), ((1, 1), 5, 256, 640), ((1, 2), 100, few, 640), ((2, 1), 16, odd, 640), ((2, 1), 5, two, short), ((2, 2), 17, odd, 640),
             ((2, 3), 48, odd, 640), ((2, 4), 64, odd, 640), ((2, 4), 128, 12416, 640), ((2, 2), 32, two, short), ((4, 1), 16, two, long), ((4, 2), 25, two, long),
             ((4, 3), 48, two, long), ((4, 4), 64, two, long), ((4, 1), 1, 16512, 640), ((4, 3), 80, 16512, 640)]
    if kind in ("mxfp8", "mxfp4"):
        cases += [((2, 6), 96, odd, short), ((4, 4), 81, odd, long), ((4, 4), 128, odd, long)]
        if kind == "mxfp4" and not row_major:
            cases += [((2, 4), 128, odd, short)]
    else:
        cases += [((2, 6), 96, two, 640), ((2, 6), 81, odd, 640)]
    if not row_major:
        cases += [((2, 3), 48, two, short)] + ([] if kind == "block" else [((2, 4), 64, two, short)])
        cases += [((2, 1), 8, 13312, long), ((4, 1), 9, 13312, long)]
    elif kind in ("fp8", "bf16"):
        cases += [((1, 1), 4, odd, 640), ((2, 1), 8, two, 1024)]
    return cases


def _reachable(kind, row_major):
    step = 128 if kind == "block" else 16
    return {routes.flat_split(kind, row_major, m, n, k) for m in (1, 4, 8, 9, 16, 32, 48, 64, 80, 96, 112, 128) for n in list(range(step, 17000, 8 * step)) + [4096, 4096 + step, 8192 + step]
            for k in (512, 1024, 2048, 4096, 8192)}


@pytest.fixture
def flat_route():
    before = g.lib().a8w8_route_override(1)      # whatever the cost model says of a case
    yield
    g.lib().a8w8_route_override(before)


@pytest.mark.parametrize("row_major", [False, True])
@pytest.mark.parametrize("kind", routes.KINDS)
def test_every_split_is_exact(kind, row_major, flat_route):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert cus == 256, "the cases are made for 256 compute units"
    assert {c[0] for c in _split_cases(kind, row_major)} == _reachable(kind, row_major)
    for split, m, n, k in _split_cases(kind, row_major):
        assert routes.flat_split(kind, row_major, m, n, k) == split, (m, n, k)
        gen = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
        if kind == "bf16":
            a, b = (torch.randint(-4, 5, (rows, k), generator=gen, device="cuda").bfloat16() for rows in (m, n))
            want = (a.double() @ b.double().T).float()
            got = g.gemm_a16w16(a, b, c_dtype=g.FP32) if row_major else g.flatmm_a16w16(a, g.preshuffle_b_bf16_device(b), n, c_dtype=g.FP32)
            assert torch.equal(got, want), (split, m, n, k)
        elif kind == "mxfp4":
            (a, sa, A), (b, sb, B) = (_mxfp4(gen, rows, k) for rows in (m, n))
            got = (g.gemm_a4w4(a, b, sa, sb, c_dtype=g.FP32) if row_major else
                   g.flatmm_a4w4(a, g.preshuffle_b_device(b), sa, sb, n, c_dtype=g.FP32))
            assert torch.equal(got, (A @ B.T).float()), (split, m, n, k)
        else:
            for mode in {"fp8": (g.TENSOR, g.ROWCOL), "block": (g.BLOCK,), "mxfp8": (g.MX_TILED,)}[kind]:
                (a, sa, A), (b, sb, B) = _scaled(gen, m, k, mode, False), _scaled(gen, n, k, mode, True)
                want = (A @ B.T).float()
                got = (g.gemm(a, b, sa, sb, mode, c_dtype=g.FP32) if row_major else
                       g.flatmm(a, g.preshuffle_b_device(b), sa, sb, n, scale_mode=mode, c_dtype=g.FP32))
                assert torch.equal(got, want), (split, mode, m, n, k)


def _mxfp4(gen, rows, k):
    value = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
    c = torch.randint(0, 16, (rows, k), generator=gen, device="cuda")
    e = torch.randint(125, 130, (rows, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
    return ((c[:, ::2] | c[:, 1::2] << 4).to(torch.uint8), g.mx_tile_scales(e),
            torch.cat([value, -value])[c] * torch.exp2(e.double() - 127).repeat_interleave(32, 1))
