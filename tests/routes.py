"""The library's size rules (gcnasm_amd/csrc/routes.hpp), loaded from tests/harness/libroutes.so: what a dispatch chooses for
given sizes, without a GPU."""
import ctypes
import os
import subprocess

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "harness")
_lib = None


def lib():
    global _lib
    if _lib is None:
        path = os.path.join(HERE, "libroutes.so")
        if not os.path.exists(path):
            subprocess.check_call(["make", "-C", HERE, "libroutes.so"], stdout=subprocess.DEVNULL)
        _lib = ctypes.CDLL(path)
    return _lib


_ll = ctypes.c_longlong


def mx_padding_in_launch(rows, k):
    return bool(lib().route_mx_padding_in_launch(_ll(rows), _ll(k)))


def quant_mx_by_lines(rows, k, fp4=False):
    """Waves per workgroup of the quantiser by lines of the tiled scales (padding in the launch), or None."""
    return (None, 4, 8)[lib().route_quant_mx_by_lines(int(fp4), _ll(rows), _ll(k))]


def quant_mx_chunks(elements, fp4=False, rows_apart=False):
    return int(lib().route_quant_mx_chunks(int(fp4), _ll(elements), int(rows_apart)))


def quant_rows_by_wave(rows, k):
    return bool(lib().route_quant_rows_by_wave(_ll(rows), _ll(k)))


def partial_steps_on_tiles(m, n, k_bytes, batch=1):
    return bool(lib().route_partial_steps_on_tiles(_ll(m), _ll(n), _ll(k_bytes), _ll(batch)))


def cvt_fnuz_few(n):
    return bool(lib().route_cvt_fnuz_few(ctypes.c_ulonglong(n)))


def quant_1x128_along_rows(rows, k):
    return bool(lib().route_quant_1x128_along_rows(_ll(rows), _ll(k)))


def f4_row_scales_on_256_tiles(m, n, k, batch=1, fp32=False, cus=256):
    """k in elements; for problems of more than two 128-tiles per compute unit whose K and scale rows the four-wave kernel takes."""
    return bool(lib().route_f4_row_scales_on_256_tiles(_ll(m), _ll(n), _ll(k // 256), _ll(batch), int(fp32), _ll(cus)))


def odd_steps_on_four_waves(steps):
    """Per-tensor and row/col scales and bf16; K steps of 128 bytes."""
    return bool(lib().route_odd_steps_on_four_waves(_ll(steps)))


def mx_row_scales_on_four_waves(steps):
    return bool(lib().route_mx_row_scales_on_four_waves(_ll(steps)))


def odd_tiled_mx_on_four_waves(m, n, steps, fp4=False, batch=1, fp32=False, cus=256):
    return bool(lib().route_odd_tiled_mx_on_four_waves(int(fp4), _ll(m), _ll(n), _ll(steps), _ll(batch), int(fp32), _ll(cus)))


KINDS = ("fp8", "block", "bf16", "mxfp8", "mxfp4")          # enum FlatKind
BYTES = {"bf16": 2.0, "mxfp4": 0.5}                          # per element of a weight row, else 1


def flat_split(kind, row_major, m, n, k, batch=1, cus=256):
    """(weight tiles, row groups) per workgroup of the flat GEMM; k in elements."""
    split = lib().route_flat_split(KINDS.index(kind), int(row_major), _ll(m), _ll(n), _ll(int(k * BYTES.get(kind, 1))), _ll(batch), _ll(cus))
    return split // 10, split % 10


def flat_is_faster(kind, row_major, m, n, k, batch=1, cus=256):
    """The flat GEMM's side of the cost model, with the layout factors of the entry points; k in elements."""
    row_bytes = int(k * BYTES.get(kind, 1))
    factor = (1.1 if kind == "mxfp8" else 1.0) * ((1.3 if row_bytes % 4096 == 0 else 1.05) if row_major else 1.0)
    return bool(lib().route_flat_is_faster(_ll(m), _ll(n), _ll(row_bytes), _ll(batch), ctypes.c_double(factor), _ll(cus)))


def rounds_on_128_tiles(m, n, steps, kind="fp8", batch=1, fp32=False, cus=256, shuffled=False):
    """kind: "fp8" (per-tensor and row/col scales), "bf16", "mxfp8", "mxfp4" (tiled scales), "block", "mx" (row-major scales)."""
    return bool(lib().route_rounds_on_128_tiles({"fp8": 0, "bf16": 0, "mxfp8": 1, "mxfp4": 2, "block": 3, "mx": 4}[kind], _ll(m), _ll(n), _ll(steps), _ll(batch), int(fp32), _ll(cus), int(shuffled)))


def narrow_tiles_deep(kind, m, k_bytes, n=1024):
    """More than three LDS stages for 128 x 64 tiles; kind as below, "mxfp8" (tiled scales), "ragged" (partial K steps)."""
    return bool(lib().route_narrow_tiles_deep(_ll(m), _ll(n), _ll(k_bytes), 0 if kind in ("fp8", "mxfp8", "bf16") else 1 if kind == "block" else 2))


def tiles_in_runs(tiles_m, tiles_n, steps, batch=1, tall=False, cus=256):
    """128-tile kernel: a run of tiles per XCD, or every eighth; tall: tiles of more rows than columns."""
    return bool(lib().route_tiles_in_runs(_ll(tiles_m), _ll(tiles_n), _ll(steps), _ll(batch), int(tall), _ll(cus)))


def items_in_runs(tiles_m, tiles_n, steps, batch=1, cus=256):
    """256-tile kernels."""
    return bool(lib().route_items_in_runs(_ll(tiles_m), _ll(tiles_n), _ll(steps), _ll(batch), _ll(cus)))


TILE128 = ("128x64", "128, four stages", "256x128", "128, two stages", "64x64")     # enum Tile128


def tile128_variant(kind, m, n, k_bytes, batch=1, cus=256, fp32=True):
    """The variant of the 128-tile kernel, or None for a problem of more than two 128-tiles per compute unit.  kind: "fp8", "mx", "block",
    "bf16", "mxfp4" (row-major scales), "mxfp4_tiled"; whole K steps.  fp32: the type of C (block scales)."""
    if not lib().route_fits_128_tiles(_ll(m), _ll(n), _ll(batch), _ll(cus)):
        return None
    return TILE128[lib().route_tile128_variant(_ll(m), _ll(n), _ll(k_bytes), _ll(batch), int(kind != "block"), int(kind in ("bf16", "mxfp4_tiled")), _ll(cus), int(kind == "block" and fp32))]
