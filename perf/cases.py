"""The work a program that uses this library has it do, as cases that can be timed and compared.

Three paths, each through the package's public functions only:

  linear   one linear layer of a quantised model: the fp32 activations of this step are quantised (their scales are
           not known before) and multiplied with weights that were quantised, and for decoding pre-shuffled, when the
           model was loaded.  `flat` cases keep the weights in the pre-shuffled layout (decoding, up to 128 tokens), the
           others row-major (prompts and batches).
  gemm     a GEMM on operands that are already in the library's formats: the bf16 sibling, and the reference-style
           program's batched block-scale GEMM with fp32 output.
  convert  fp32 -> E4M3 -> fp32 through the bit-exact conversion helpers (a cache or a checkpoint shard written and
           read back).

A case is a dict of plain values; m, n, k are tokens, output features and input features.  `out` is the type of C.
"""
import math

import torch

import gcnasm_amd as g

SCALES = {"tensor": g.TENSOR, "rowcol": g.ROWCOL, "block": g.BLOCK, "mx": g.MX, "mx_tiled": g.MX_TILED}


def _case(path, mode, m, n, k, out="bf16", flat=False, batch=1, **more):
    return dict(path=path, mode=mode, m=m, n=n, k=k, out=out, flat=flat, batch=batch, **more)


def listed():
    cases = {
        # one token of one sequence through a small layer: launches and the host's part count as much as the kernels
        "decode_rowcol_1x4096x4096": _case("linear", "rowcol", 1, 4096, 4096, flat=True),
        # a decoding batch of 16 over a wide layer: the weight stream from HBM
        "decode_rowcol_16x16384x7168": _case("linear", "rowcol", 16, 16384, 7168, flat=True),
        # a large decoding batch, MXFP8: the activations are re-read by every workgroup
        "decode_mx_tiled_64x16384x7168": _case("linear", "mx_tiled", 64, 16384, 7168, flat=True),
        # a prefill chunk of 256 tokens: too many rows for the flat kernel, too few for the large tiles
        "chunk_rowcol_256x8192x8192": _case("linear", "rowcol", 256, 8192, 8192),
        # sizes that are no multiple of any tile, K step or group of 16 rows
        "ragged_rowcol_1000x3000x2000": _case("linear", "rowcol", 1000, 3000, 2000),
        # per-tensor scales, a mid-sized square problem between the tile sizes
        "prefill_tensor_2560x2560x2560": _case("linear", "tensor", 2560, 2560, 2560),
        # 1x128 / 128x128 block scales, a prompt of 4096 tokens
        "prefill_block_4096x7168x2048": _case("linear", "block", 4096, 7168, 2048),
        # MXFP4 with the scales as the quantiser writes them by default (row-major)
        "prefill_mxfp4_4096x4096x4096": _case("linear", "mxfp4", 4096, 4096, 4096),
        # the largest: a long prompt in MXFP8
        "prefill_mx_tiled_8192x8192x8192": _case("linear", "mx_tiled", 8192, 8192, 8192),
        # layers that stay in bf16
        "gemm_bf16_4096x4096x4096": _case("gemm", "bf16", 4096, 4096, 4096),
        # the reference-style program with a batch: fp32 output, one problem per expert or head
        "gemm_block_8x512x1024x1024": _case("gemm", "block", 512, 1024, 1024, out="fp32", batch=8),
        # conversions both ways, 4096 x 8192 values
        "convert_ocp_clamp_32M": _case("convert", "ocp", 4096, 8192, 1, out="fp32", clamp=True),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _spread(rng, low, high, step):
    """A multiple of `step` between low and high, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high, max(low, int(round(v / step)) * step))


def draw(rng):
    family = rng.choice(["decode", "decode", "linear", "linear", "linear", "gemm", "convert"])
    if family == "decode":
        # weights in the pre-shuffled layout: whole groups of 16 rows and of 64 columns (block and MX scales: 128)
        mode = rng.choice(["rowcol", "rowcol", "tensor", "block", "mx_tiled", "mxfp4_tiled"])
        step_n = 128 if mode == "block" else 16
        step_k = {"rowcol": 64, "tensor": 64}.get(mode, 128)
        m, n, k = _spread(rng, 1, 128, 1), _spread(rng, 1024, 28672, step_n), _spread(rng, 1024, 8192, step_k)
        return _case("linear", mode, m, n, k, flat=True)
    if family == "linear":
        mode = rng.choice(["rowcol", "rowcol", "tensor", "block", "mx", "mx_tiled", "mxfp4", "mxfp4_tiled"])
        m = _spread(rng, 129, 8192, 1)
        n, k = _spread(rng, 512, 8192, 128), _spread(rng, 512, 8192, 256)
        if mode in ("rowcol", "tensor"):
            ragged = rng.choice([False, False, True])
            n = _spread(rng, 512, 8192, 4 if ragged else 64)
            k = _spread(rng, 512, 4096, 16) if ragged else _spread(rng, 512, 8192, 128)
            if ragged:
                m = min(m, 2048)
        elif mode in ("mx", "mx_tiled"):
            k = _spread(rng, 512, 8192, 128)
        return _case("linear", mode, m, n, k, out=rng.choice(["bf16", "bf16", "fp32"]))
    if family == "gemm":
        mode = rng.choice(["bf16", "block"])
        batch = rng.choice([1, 1, 2, 4, 8, 16])
        top = 4096 if batch <= 2 else 1024
        m, n, k = _spread(rng, 64, top, 1), _spread(rng, 256, top, 128), _spread(rng, 256, 4096, 128)
        return _case("gemm", mode, m, n, k, out=rng.choice(["bf16", "fp32"]), batch=batch)
    rows, cols = _spread(rng, 64, 8192, 1), _spread(rng, 256, 8192, 1)
    return _case("convert", rng.choice(["ocp", "ocp", "fnuz"]), rows, cols, 1, out="fp32", clamp=rng.choice([True, False]))


# ------------------------------------------------------------------ inputs
def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _activations(gen, rows, k, mode):
    """N(0, 1); for the MX formats each block of 32 has a magnitude of its own, as it has where those formats are used."""
    x = torch.randn((rows, k), generator=gen, device="cuda")
    if mode.startswith("mx") and k % 32 == 0:
        x.view(rows, k // 32, 32).mul_(torch.exp2(torch.rand((rows, k // 32, 1), generator=gen, device="cuda") * 8 - 4))
    return x


def _quantize(x, mode, weight):
    if mode == "mxfp4":
        return g.quantize_mxfp4(x)
    if mode == "mxfp4_tiled":
        return g.quantize_mxfp4(x, tiled=True)
    return g.quantize(x, SCALES[mode], group_rows=128 if weight and mode == "block" else 1)


def _c_dtype(case):
    return g.FP32 if case["out"] == "fp32" else g.BF16


def prepare(case, seed):
    gen = _generator(seed)
    m, n, k, mode, batch = case["m"], case["n"], case["k"], case["mode"], case["batch"]
    state = dict(case=case, c_dtype=_c_dtype(case))
    if case["path"] == "convert":
        state["x"] = torch.randn((m, n), generator=gen, device="cuda") * 64.0      # a few beyond 240: the clamp has work
        state["dialect"] = g.FNUZ if mode == "fnuz" else g.OCP
    elif case["path"] == "linear":
        state["x"] = _activations(gen, m, k, mode)
        w, state["w_scale"] = _quantize(_activations(gen, n, k, mode), mode, weight=True)
        state["w"] = g.preshuffle_b_device(w) if case["flat"] else w
    elif mode == "bf16":
        shape = (lambda rows: (batch, rows, k)) if batch > 1 else (lambda rows: (rows, k))
        state["a"] = torch.randn(shape(m), generator=gen, device="cuda").to(torch.bfloat16)
        state["b"] = torch.randn(shape(n), generator=gen, device="cuda").to(torch.bfloat16)
    else:
        a = [_quantize(_activations(gen, m, k, mode), mode, weight=False) for _ in range(batch)]
        b = [_quantize(_activations(gen, n, k, mode), mode, weight=True) for _ in range(batch)]
        pick = (lambda pairs, i: torch.stack([p[i] for p in pairs])) if batch > 1 else (lambda pairs, i: pairs[0][i])
        state.update(a=pick(a, 0), b=pick(b, 0), sfa=pick(a, 1), sfb=pick(b, 1))
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    mode = case["mode"]
    if case["path"] == "convert":
        codes = g.cvt_f32_to_e4m3(state["x"], state["dialect"], clamp240=case["clamp"])
        return codes, g.cvt_e4m3_to_f32(codes, state["dialect"])
    if case["path"] == "gemm":
        if mode == "bf16":
            return g.gemm_a16w16(state["a"], state["b"], c_dtype=state["c_dtype"])
        return g.gemm_blockscale(state["a"], state["b"], state["sfa"], state["sfb"], c_dtype=state["c_dtype"])
    q, scale = _quantize(state["x"], mode, weight=False)
    w, w_scale, c_dtype, n = state["w"], state["w_scale"], state["c_dtype"], case["n"]
    if mode.startswith("mxfp4"):
        if case["flat"]:
            return g.flatmm_a4w4(q, w, scale, w_scale, n, c_dtype=c_dtype)
        return g.gemm_a4w4(q, w, scale, w_scale, g.MX if mode == "mxfp4" else g.MX_TILED, c_dtype=c_dtype)
    if case["flat"]:
        return g.flatmm(q, w, scale, w_scale, n, scale_mode=SCALES[mode], c_dtype=c_dtype)
    return g.gemm(q, w, scale, w_scale, SCALES[mode], c_dtype=c_dtype)


# ------------------------------------------------------------------ what a pass cannot do without
def _scale_bytes(mode, rows, k, weight):
    if mode == "tensor":
        return 4
    if mode == "rowcol":
        return 4 * rows
    if mode == "block":
        return 4 * (k // 128) * (rows // 128 if weight else rows)
    return rows * (k // 32) if mode.startswith("mx") else 0


def work(case):
    m, n, k, mode, batch = case["m"], case["n"], case["k"], case["mode"], case["batch"]
    if case["path"] == "convert":
        return {"bytes": m * n * (4 + 1 + 1 + 4), "flops": 0}
    element = 2.0 if mode == "bf16" else 0.5 if mode.startswith("mxfp4") else 1.0
    out = m * n * (4 if case["out"] == "fp32" else 2)
    weights = n * k * element + _scale_bytes(mode, n, k, True)
    if case["path"] == "linear":
        inputs = m * k * 4.0                # the fp32 activations; their quantised form is the pass's own
    else:
        inputs = m * k * element + _scale_bytes(mode, m, k, False)
    return {"bytes": int(batch * (inputs + weights + out)), "flops": 2 * batch * m * n * k}


def tolerance(case):
    """Conversions are exact, and so are the quantised operands of a GEMM; what is left is the order and width of the
    accumulation and the rounding of C.  The bounds are four times what the GEMMs were seen to differ by from float64
    products of the same operands (512^3 to 700 x 1024 x 4096 and 8 .. 300 x 2048 x 7168, every scale mode):
      bf16 C   against the rounded float64 value: 2.4e-4 in norm, never more than one unit in the last place (7.8e-3)
      fp32 C   FP8 operands 1.5e-5 and at most 3.5e-4 (the FP8 matrix instruction aligns its 128 products to the largest
               one), bf16 operands 4e-7 and 2.8e-6, FP4 operands 2e-8 and 2.4e-7 (fp32 sums in another order: up to ten
               times that)"""
    if case["path"] == "convert":
        return "exact"
    if case["out"] == "bf16":
        return {"rel": 1e-3, "max": 1.6e-2}
    if case["mode"] == "bf16" or case["mode"].startswith("mxfp4"):
        return {"rel": 1.6e-6, "max": 1.2e-5}
    return {"rel": 6e-5, "max": 1.4e-3}
