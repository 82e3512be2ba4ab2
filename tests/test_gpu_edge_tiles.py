"""Edge tiles of the 128-tile kernel: where the matrix ends on a 16-byte piece of a row they leave through LDS like whole tiles,
elsewhere element by element.  C lies inside a sentinel-filled array, so a store outside it shows; operands are exact."""
import pytest
import torch

import gcnasm_amd as g

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 16, 65, 129, 250, 256])
@pytest.mark.parametrize("n", [8, 60, 72, 136, 252, 1000])
@pytest.mark.parametrize("k", [256, 2048, 272])               # wide tiles, narrow tiles, a partial K step
@pytest.mark.parametrize("mode", [g.TENSOR, g.ROWCOL])
def test_nothing_outside_the_matrix(m, n, k, mode):
    gen = torch.Generator(device="cuda").manual_seed(m * 1009 + n + k)
    a, b = (torch.randint(-4, 5, (rows, k), generator=gen, device="cuda").float() for rows in (m, n))
    sa, sb = (torch.exp2(torch.randint(-2, 3, (rows if mode == g.ROWCOL else 1,), generator=gen, device="cuda").float()) for rows in (m, n))
    ref = (a.double() * sa[:, None]) @ (b.double() * sb[:, None]).T
    for c_dtype, dtype in ((g.BF16, torch.bfloat16), (g.FP32, torch.float32)):
        whole = torch.full((m + 3, n + 24 - n % 8), 7.0, dtype=dtype, device="cuda")
        whole[:m, :n] = float("nan")
        g.gemm(g.cvt_f32_to_e4m3(a), g.cvt_f32_to_e4m3(b), sa, sb, mode, c=whole[:m, :n])
        assert torch.equal(whole[:m, :n], ref.to(torch.float32).to(dtype))
        assert (whole[m:] == 7.0).all() and (whole[:, n:] == 7.0).all()
