// The library's size rules (gcnasm_amd/csrc/routes.hpp) behind C functions, for the tests.
#include "../../gcnasm_amd/csrc/routes.hpp"

extern "C" {
int route_mx_padding_in_launch(long long rows, long long k) { return a8w8::mx_padding_in_launch(rows, k); }
int route_quant_mx_by_lines(int fp4, long long rows, long long k) { return a8w8::quant_mx_by_lines(fp4 != 0, rows, k); }
int route_quant_mx_chunks(int fp4, long long elements, int rows_apart) { return a8w8::quant_mx_chunks(fp4 != 0, elements, rows_apart != 0); }
int route_quant_rows_by_wave(long long rows, long long k) { return a8w8::quant_rows_by_wave(rows, k); }
int route_partial_steps_on_tiles(long long m, long long n, long long k_bytes, long long batch)
{
    return a8w8::partial_steps_on_tiles(m, n, k_bytes, batch);
}
int route_cvt_fnuz_few(unsigned long long n) { return a8w8::cvt_fnuz_few(n); }
int route_quant_1x128_along_rows(long long rows, long long k) { return a8w8::quant_1x128_along_rows(rows, k); }
int route_f4_row_scales_on_256_tiles(long long m, long long n, long long k_steps, long long batch, int fp32_c, long long cus)
{
    return a8w8::f4_row_scales_on_256_tiles(m, n, k_steps, batch, fp32_c != 0, cus);
}
int route_odd_steps_on_four_waves(long long k_steps) { return a8w8::odd_steps_on_four_waves(k_steps); }
int route_mx_row_scales_on_four_waves(long long k_steps) { return a8w8::mx_row_scales_on_four_waves(k_steps); }
int route_odd_tiled_mx_on_four_waves(int fp4, long long m, long long n, long long k_steps, long long batch, int fp32_c, long long cus)
{
    return a8w8::odd_tiled_mx_on_four_waves(fp4 != 0, m, n, k_steps, batch, fp32_c != 0, cus);
}
// 10 nt + mt
int route_flat_split(int kind, int row_major, long long m, long long n, long long row_bytes, long long batch, long long cus)
{
    const a8w8::FlatSplit f = a8w8::flat_split((a8w8::FlatKind)kind, row_major != 0, m, n, row_bytes, batch, cus);
    return 10 * f.nt + f.mt;
}
int route_flat_is_faster(long long m, long long n, long long row_bytes, long long batch, double layout_factor, long long cus)
{
    return a8w8::flat_is_faster(m, n, row_bytes, batch, layout_factor, cus);
}
int route_rounds_on_128_tiles(int kind, long long m, long long n, long long k_steps, long long batch, int fp32_c, long long cus, int b_shuffled)
{
    return a8w8::rounds_on_128_tiles((a8w8::RoundsKind)kind, m, n, k_steps, batch, fp32_c != 0, cus, b_shuffled != 0);
}
int route_narrow_tiles_deep(long long m, long long n, long long k_bytes, int kind) { return a8w8::narrow_tiles_deep(m, n, k_bytes, (a8w8::StepKind)kind); }
int route_tiles_in_runs(long long tiles_m, long long tiles_n, long long k_steps, long long batch, int tall, long long cus)
{
    return a8w8::tiles_in_runs(tiles_m, tiles_n, k_steps, batch, tall != 0, cus);
}
int route_items_in_runs(long long tiles_m, long long tiles_n, long long k_steps, long long batch, long long cus)
{
    return a8w8::items_in_runs(tiles_m, tiles_n, k_steps, batch, cus);
}
int route_fits_128_tiles(long long m, long long n, long long batch, long long cus) { return a8w8::fits_128_tiles(m, n, batch, cus); }
int route_tile128_variant(long long m, long long n, long long k_bytes, long long batch, int has_tall, int cheap_steps, long long cus, int block_fp32)
{
    return a8w8::tile128_variant(m, n, k_bytes, batch, has_tall != 0, cheap_steps != 0, cus, block_fp32 != 0);
}
}
