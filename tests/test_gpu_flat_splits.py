"""How the flat GEMM deals weight tiles and row groups to workgroups: every split its rule can choose (layers from a few
weight tiles to more than two per compute unit, two to eight groups of 16 rows, ragged last ones), against exact products, on
pre-shuffled and on row-major weights."""
import pytest
import torch

import gcnasm_amd as g

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
