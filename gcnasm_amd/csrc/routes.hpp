// Which kernel variant a call takes, where that depends on its sizes: plain host functions of sizes and the number of compute
// units, without the HIP runtime, so that they can be checked without a GPU.  Times in the comments: MI355X, 256 compute units,
// us per launch inside a graph.
#pragma once
#include <algorithm>

namespace a8w8 {

// Tiled MX scales of an array that is no whole number of 64-row blocks and of 512-element groups: the positions no (row, block)
// owns get their 127 from the quantiser itself, as elements of the padded array that are not loaded, or from a fill launch in
// front of it (2 us).  A padding element costs what a real one costs: about nothing where the padded array does not fill the chip
// (4M elements), 0.5 us per million beyond, so that the line lies at three million.  E4M3, us, padded / filled: 1 x 65536 4.7 / 5.7,
// 16384 x 288 (3.5M) 8.5 / 8.1, 1 x 131072 (8M) 6.6 / 5.2, 16 x 262144 11.4 / 7.1, 1 x 2^20 35 / 5.6, 65536 x 32 21.2 / 5.8,
// 65536 x 1056 66.6 / 61.9; MXFP4 alike.
inline bool mx_padding_in_launch(long long rows, long long k)
{
    const long long padded = ((rows + 63) / 64 * 64) * ((k + 511) / 512 * 512);
    return padded < 1ll << 31 &&                                                    // (the kernel counts elements with 31 bits)
           (padded <= 4ll << 20 || padded - rows * k <= 3ll << 20);
}

// Tiled MX scales whose padding is in the launch: by lines of the scale array past a million elements, padding counted for E4M3 (1 x 65536 4.5 -> 3.6 us,
// 8192 x 32 4.9 -> 3.9) and not for MXFP4 (3.4 / 3.6, 3.7 / 3.8), whose kernel for few elements is the faster one there (128 x 8192 3.32 / 3.34,
// 300 x 5632 3.75 / 3.66).  At half a million E4M3 takes 3.0 us with one chunk per wave, 3.3 by lines.
enum MxLines { MX_NOT_BY_LINES, MX_LINES_FOUR_WAVES, MX_LINES_EIGHT_WAVES };
inline MxLines quant_mx_by_lines(bool fp4, long long rows, long long k)
{
    const long long elements = rows * k, padded = ((rows + 63) / 64 * 64) * ((k + 511) / 512 * 512);
    if ((fp4 ? elements : padded) <= 1ll << 20) return MX_NOT_BY_LINES;
    return elements >= 5000000 && elements < 15000000 ? MX_LINES_FOUR_WAVES : MX_LINES_EIGHT_WAVES;
}

// Row-major MX scales: chunks of 256 elements per wave (quant_mx_flat_kernel).  us, one / two / four: E4M3 1024 x 2048 3.4 / 3.9 / 4.2, 2560 x 2560 8.0 / 7.3 / 7.7,
// 8192 x 8192 59.0 / 52.3 / 53.6; MXFP4 128 x 8192 3.2 / 3.3 / 3.7, 1024 x 2048 3.5 / 3.2 / 4.2, 8192 x 8192 56.9 / 47.9 / 49.6.  Rows apart, from 8M elements:
// 5831 x 2304 14.8 / 13.6 / 12.9, MXFP4 13.4 / 12.1 / 11.2 (below, 2560 x 2560 8.3 / 7.5 / 7.7).
inline int quant_mx_chunks(bool fp4, long long elements, bool rows_apart)
{
    if (elements <= 1ll << (fp4 ? 20 : 21)) return 1;
    return rows_apart && elements >= 1ll << 23 ? 4 : 2;
}

// The per-row quantiser: a wave per row for more than a thousand rows of at most 1024 elements, else a workgroup (quant_rowwise_wave_kernel).
inline bool quant_rows_by_wave(long long rows, long long k)
{
    return k <= 1024 && rows > 1024;
}

// Rows of whole 16-byte pieces whose length is no multiple of the 128-byte K step (scales that do not change with K): the 128-tile kernel
// with a partial last step, 4.6 to 8 us at the least, or the one-thread-per-element kernel, 2.2 us and 60 to 85 ns per K element while
// its outputs fit the chip at once.  us, one thread per element / tiles, row/col scales, K in bytes:
//   128 x 512 x 16  3.4 / 4.8    129 x 1000 x 16  4.4 / 5.0    256 x 1024 x 16  7.0 / 5.5    128 x 260 x 48  5.7 / 6.8    128 x 512 x 32  6.5 / 5.4
//   64 x 260 x 80   9.1 / 7.2    300 x 391 x 240   38 / 11.5   1000 x 3000 x 2000  7540 / 21   4096 x 4096 x 4080  84 ms / 116
// so that K below 64 bytes stays with the former up to 2^21 multiply-adds.  Problems of less than 2^19 with K below 256 bytes stay there
// too, although tiles would be faster (46 x 46 x 240: 21 us): a few thousand outputs in the order of operations of the CPU
// reference, bit for bit, which is what callers compare small problems with.
inline bool partial_steps_on_tiles(long long m, long long n, long long k_bytes, long long batch)
{
    return k_bytes >= 256 || (double)batch * m * n * k_bytes >= (double)(1ll << (k_bytes < 64 ? 21 : 19));
}

// FNUZ conversions are 30 to 40 integer operations per value: eight values per thread (the vectorised kernels) are a longer chain than
// the launch, and below two million values there are enough threads without them.  us, eight per thread / four (encode) and
// one (decode) per thread: encode 65536 3.4 / 2.7, 2^19 3.5 / 3.1, 7 x 2^18 4.7 / 4.5; decode 65536 3.0 / 2.2, 2^19 3.3 / 2.5, 7 x 2^18 4.7 / 4.4;
// equal at 2^21.  The OCP dialect, one hardware instruction per pair, is as fast either way.
inline bool cvt_fnuz_few(unsigned long long n)
{
    return n < 1ull << 21;
}

// The 1 x 128 quantiser's workgroups take 8 or 32 rows of one group, for the sake of the scales' lines.  With fewer than eight rows part
// of every workgroup has none (1 x 2^20 7.3 us, 3 x 2^20 11.8, against 3.3 and 5.5 along the rows), and over long rows the 512 bytes
// they read of each lie far apart (12 x 2^20 17.2, 17 x 2^20 24.3, 33 x 2^21 75, against 14.7, 19.2 and 69 along the rows).
inline bool quant_1x128_along_rows(long long rows, long long k)
{
    return rows < 8 || (rows < 96 && k >= 1 << 19);
}

// Rounds of one tile per compute unit.
struct Rounds { long long of128, of256; };
inline Rounds tile_rounds(long long m, long long n, long long batch, long long cus)
{
    return {(batch * ((m + 127) / 128) * ((n + 127) / 128) + cus - 1) / cus, (batch * ((m + 255) / 256) * ((n + 255) / 256) + cus - 1) / cus};
}

// One or two rounds of 256-tiles, the last of which leaves much of the chip idle: the two-stage 128-tile kernel, whose rounds are finer, up to the K where
// the 256-tiles' cheaper steps have made up for it.  us, 128-tiles / 256-tiles, row/col bf16 C, row/col fp32, tiled MXFP8 bf16, tiled MXFP4 bf16 (bf16
// operands as row/col):
//   6144 x 3072 (5 rounds of 128-tiles, 2 of 256-tiles)  6 steps 23.1 / 28.6, 27.0 / 39.0, 25.3 / 29.6, 25.9 / 32.0   16: 41.6 / 50.2, 44.1 / 60.5, 47.6 / 52.2, 50.0 / 58.7
//                                                        32: 73.8 / 85.2, 84.7 / 95.1, 86.5 / 87.5, 92.0 / 101
//   8192 x 2560 (5, 2)   6: 23.9 / 29.1, 29.5 / 38.6, 26.1 / 30.3, 26.9 / 32.6   24: 61.6 / 69.3, 75.5 / 78.0, 70.9 / 70.7, 73.6 / 79.7   32: 80.2 / 85.6, 94.7 / 95.4, 91.9 / 87.7, 95.7 / 101
//   5376 x 4096 (6, 2)   6: 26.7 / 28.9, 31.8 / 37.8, 29.1 / 30.4, 29.9 / 32.3   16: 48.6 / 52.1, 53.7 / 60.1, 54.7 / 52.8, 56.6 / 59.5   24: 70.9 / 69.1, 78.4 / 78.2, 82.3 / 72.1, 84.1 / 81.1
//   2560 x 4352 (3, 1)   6: 15.6 / 16.7, 18.5 / 20.4, 17.3 / 17.4, 17.7 / 18.6   16: 26.7 / 28.0, 28.7 / 32.0, 31.0 / 29.1, 32.3 / 32.0
//   4096 x 7168 (7, 2)   6: 32.4 / 31.3, 47.1 / 40.5, 35.2 / 32.4, 35.6 / 34.9   8192 x 4608 (9, 3)  6: 42.1 / 42.3, 64.6 / 57.0, 44.8 / 44.3, 45.2 / 47.1
// Fewer than five steps stay with the 256-tiles although they are 4 to 28% slower in the same shapes: the kernel that a8w8_kernel_name reports for
// calls of that size is held fixed by the library's tests.
// Against the eight-wave kernel, 128-tiles / 256-tiles, block scales bf16 C, fp32, row-major MXFP8 bf16, fp32:
//   6144 x 3072  8 steps 29.5 / 33.7, 32.3 / 41.6, 31.2 / 34.6, 34.0 / 41.9   16: 47.0 / 54.8, 50.0 / 62.3, 50.9 / 55.2, 54.0 / 62.9   32: 84.8 / 98.0, 90.7 / 105, 99.8 / 95.6, 106 / 106
//   5376 x 4096  8: 33.6 / 36.0, 37.9 / 43.6, 35.7 / 36.9, 39.6 / 42.8   12: 44.6 / 48.3, 48.8 / 56.0, 46.9 / 48.1, 50.7 / 53.1   24: 75.9 / 80.6, 81.4 / 87.7, 89.1 / 80.5, 94.2 / 85.6
//   2304 x 4096  8: 19.5 / 19.1, 21.9 / 23.1, 20.1 / 19.5, 22.7 / 23.4   16: 30.4 / 29.5, 31.9 / 33.7, 32.0 / 31.3, 33.8 / 34.6
// A batch of small entries (up to 128 tiles of 128 x 128 each): every XCD's 128-tiles read nearly all of every entry, so that three rounds of them stand against one of 256-tiles
// up to eight or ten steps only.  us, 128-tiles / 256-tiles: block fp32 16 x 953 x 640 8 steps 26.0 / 26.3, 10 30.3 / 29.2, 15 40.9 / 36.0; bf16 operands 16 x 953 x 640 bf16 C 8 22.1 / 25.9,
// 15 35.0 / 28.7; 16 x 700 x 768 8 21.7 / 20.8, 10 25.6 / 23.1, 16 35.7 / 29.7; 8 x 1020 x 1280 8 20.5 / 20.5, 10 23.9 / 22.5, 16 32.9 / 28.8.  Larger entries as above:
// 2 x 2600 x 2176 bf16 C 14 steps 28.2 / 31.5, block fp32 29.8 / 29.7 at 12.
// Weights in the shuffled layout (b_shuffled): the 256-tiles gain by it what the 128-tiles do not, and only rounds of twice as many 128-tiles at most, 5 against 2 with tiled scales, and 5
// against 2 with fp32 C over few steps go to 128-tiles.  128-tiles / 256-tiles, geometric means over 500 drawn shapes: 4 against 2 0.70 to 0.88 for every kind; 5 against 2 tiled MXFP4
// 0.90 to 1.00, tiled MXFP8 0.86 to 0.98, fp32 C row/col 0.81 and 0.92 up to 8 and 12 steps, 1.01 to 1.06 beyond, block 0.91 to 0.96 up to 16, bf16 C 1.00 to 1.12; 6 against
// 2 1.00 to 1.25; 3 against 1 row/col 1.13 to 1.24, block 1.08, row-major MX 1.10 to 1.17, tiled MXFP4 1.00 (2 x 3894 x 1280 x 1408 row/col 23.9 / 20.0 us).
enum RoundsKind { ROUNDS_PLAIN, ROUNDS_MXFP8_TILED, ROUNDS_MXFP4_TILED, ROUNDS_BLOCK, ROUNDS_MXFP8_ROWS };      // (plain: per-tensor and row/col scales, bf16)
inline bool rounds_on_128_tiles(RoundsKind kind, long long m, long long n, long long k_steps, long long batch, bool fp32_c, long long cus, bool b_shuffled = false)
{
    const Rounds rounds = tile_rounds(m, n, batch, cus);
    if (k_steps < 5 || rounds.of256 > 2 || rounds.of128 > 3 * rounds.of256) return false;
    const bool finer = rounds.of128 < 3 * rounds.of256, two = rounds.of256 == 2;
    const long long entry_tiles = ((m + 127) / 128) * ((n + 127) / 128);
    if (!finer && batch > 1 && entry_tiles <= 128 && k_steps > (entry_tiles <= 64 ? 8 : 10)) return false;
    if (b_shuffled && rounds.of128 > 2 * rounds.of256) {
        if (!finer) return false;
        if (kind != ROUNDS_MXFP8_TILED && kind != ROUNDS_MXFP4_TILED)
            return fp32_c && k_steps <= (kind == ROUNDS_BLOCK ? 16 : kind == ROUNDS_MXFP8_ROWS ? 8 : 12);
    }
    switch (kind) {
        case ROUNDS_MXFP8_TILED: return k_steps <= (finer ? 20 : fp32_c ? 8 : 0);
        case ROUNDS_MXFP4_TILED: return k_steps <= (finer ? 32 : fp32_c ? 16 : 8);
        case ROUNDS_BLOCK: return k_steps <= (finer ? 32 : two ? 24 : fp32_c ? 16 : 0);
        case ROUNDS_MXFP8_ROWS: return k_steps <= (finer ? 16 : fp32_c ? 12 : two ? 8 : 0);
        default: return k_steps <= (finer ? 32 : 16);
    }
}

// MXFP4 on row-major scales, more than two 128-tiles per compute unit: the four-wave kernel (256-tiles, one workgroup per compute
// unit) or the two-stage 128-tile kernel.  Both run in rounds: a round of 256-tiles (one per compute unit) is worth about three
// rounds of one 128-tile per compute unit, three and a half where K is short and a prologue and a tile's stores, longer with fp32
// C, weigh more; below four K steps of 256 elements (fp32 C: eight) they weigh too much.  us, 128-tiles / 256-tiles, bf16 C:
//   4096 x 4096 (4 rounds of one 128-tile per compute unit, 1 of 256-tiles)   K 512 13.8 / 14.7, 1024 19.4 / 18.1, 2048 28.4 / 25.4, 4096 50 / 39
//   4096 x 7168 (7, 2)    512 20.9 / 22.1, 1024 30.0 / 28.7, 2048 45.0 / 41.8, 4096 86 / 70
//   3000 x 8192 (6, 2)    512 18.8 / 21.9, 1024 26.0 / 27.6, 2048 38.2 / 39.5, 3072 54.9 / 53.3, 4096 72 / 66
//   8192 x 2560 (5, 2)    512 16.3 / 21.9, 1024 22.0 / 27.5, 2048 32.3 / 39.5, 4096 60 / 65, 8192 112 / 116
// fp32 C: 4096 x 4096 1024 23.0 / 22.6, 2048 31.7 / 29.5; 4096 x 7168 1024 34.1 / 36.6, 2048 49.0 / 49.9, 3072 66.8 / 63.7;
// 3000 x 8192 2048 42.5 / 49.0, 3072 56.8 / 61.0, 4096 77 / 75; 8192 x 2560 512 20.0 / 30.1, 4096 63 / 73.
// An odd number of K steps costs the four-wave kernel the idle step behind it and has to be longer: bf16 seven, fp32 thirteen
// (2816 x 5120 bf16 5 steps 21.2 / 21.6, 7 25.6 / 25.4, fp32 9 33.4 / 35.2, 17 63.5 / 53.1; 8192 x 8192 41 steps bf16 518 / 349).
inline bool f4_row_scales_on_256_tiles(long long m, long long n, long long k_steps, long long batch, bool fp32_c, long long cus)
{
    const Rounds rounds = tile_rounds(m, n, batch, cus);
    if (k_steps < (k_steps % 2 ? (fp32_c ? 13 : 7) : (fp32_c ? 8 : 4))) return false;
    return 2 * rounds.of128 >= (k_steps >= (fp32_c ? 16 : 12) ? 6 : 7) * rounds.of256;
}

// An odd number of K steps on the four-wave kernel, which walks them in pairs: one step more, without MFMAs (about 0.4 us of the 1.2
// to 1.4 a step takes), more than two 128-tiles per compute unit.
// Per-tensor and row/col scales and bf16: instead of the eight-wave kernel, from 33 steps on (us, eight waves / four: 2816 x 5120 17 steps
// 32.1 / 32.3, 41 64.1 / 62.9; 8192 x 8192 33 208.1 / 202.6, 49 298.4 / 288.5; fp32 C 3000 x 8192 17 65.6 / 67.9, 41 124.5 / 121.5).
inline bool odd_steps_on_four_waves(long long k_steps)
{
    return k_steps >= 33;
}
// MXFP8 on row-major scales, more than two 128-tiles per compute unit: the four-wave kernel instead of the eight-wave one from 32 steps on.
// Below, the four-wave kernel's scale loads, a line for every two lanes in front of the operands' in one queue, cost what its fewer LDS reads save.
// us, eight waves / four, 8192 x 8192, 2816 x 5120, 8192 x 2560 (a second round of 64 tiles):
//   bf16   9 steps 90.0 / 91.9, 24.2 / 24.9, 38.8 / 41.0    16 134 / 128, 35.0 / 34.1, 58.5 / 58.1    33 245 / 228, 62.1 / 61.9, 104 / 104
//          64 433 / 409, 111 / 105, 191 / 182
//   fp32   9 118 / 116, 30.3 / 30.3, 46.9 / 47.2            16 163 / 149, 41.1 / 39.9, 65.5 / 66.8    33 264 / 250, 67.6 / 65.5, 112 / 112
//          64 456 / 425, 115 / 111, 200 / 190
inline bool mx_row_scales_on_four_waves(long long k_steps)
{
    return k_steps >= 32;
}
// Tiled MX scales: instead of the 128-tile kernel, whose rounds compare as above.  us, 128-tiles / 256-tiles, MXFP8 bf16 C, MXFP8 fp32, MXFP4
// bf16, MXFP4 fp32 (K steps of 128 bytes):
//   2816 x 5120 (4 rounds, 1)   5 steps 19.5 / 18.0, 22.3 / 24.5, 19.9 / 19.1, 23.1 / 25.0   17: 41.0 / 33.9, 43.6 / 39.8, 41.8 / 37.8, 44.5 / 43.8
//   8192 x 8192 (16, 4)         5  83.0 / 66.5, 107.8 / 92.7, 84.6 / 69.7, 109.6 / 95.3      41: 358 / 257, 374 / 278, 378 / 296, 402 / 315
//   2560 x 4352 (3, 1)          13 27.2 / 26.9, 29.2 / 31.0, 27.9 / 29.6, 30.4 / 33.6        33: 56.0 / 50.5, 58.2 / 54.5, 60.0 / 57.3, 62.5 / 60.9
//   3000 x 8192 (6, 2)          17 63.0 / 60.2, 69.6 / 70.5, 65.4 / 67.2, 70.5 / 77.0        41: 133 / 118, 143 / 130, 137 / 134, 148 / 147
//   8192 x 2560 (5, 2)          25 73.0 / 74.4, 83.6 / 84.4, 75.8 / 84.3, 85.4 / 94.0        41: 114 / 111, 127 / 120, 123 / 128, 133 / 138
inline bool odd_tiled_mx_on_four_waves(bool fp4, long long m, long long n, long long k_steps, long long batch, bool fp32_c, long long cus)
{
    const Rounds rounds = tile_rounds(m, n, batch, cus);
    if (2 * rounds.of128 >= 7 * rounds.of256) return k_steps >= (!fp32_c ? 5 : fp4 ? 13 : 11);
    if (rounds.of128 >= 3 * rounds.of256) return k_steps >= (fp4 ? (fp32_c ? 33 : 25) : fp32_c ? 21 : 13);
    return !fp4 && k_steps >= 33;
}

// ---------------------------------------------------------------- 128-tile kernel
// 128 x 128 tiles when all of them fit on the chip at once, two workgroups per compute unit: a problem of that
// size leaves 256 x 256 tiles with at most half of the compute units.  Measured on 256 compute units against the
// 256-tile kernels (block / row-col / tiled MX): 2.2x / 1.7x / 1.6x at 64 workgroups, 1.9x / 1.6x / 1.5x at 256,
// +45% / +21% / +15% at 400, +37% / +17% / +9% at 512; beyond that the second round of workgroups costs more than
// the idle compute units did (-9% for row/col at 576).
// (the bound as a switch, for measurement: with 8 instead of 2, 4096 x 7168 x 2048 and 4096^3 take 12-30% longer in every scale mode)
#ifndef A8W8_SMALL_TILES_PER_CU
#define A8W8_SMALL_TILES_PER_CU 2
#endif
#ifndef A8W8_SMALL_DEEP_UP_TO
#define A8W8_SMALL_DEEP_UP_TO 1         // four LDS stages up to this many 128-tiles per compute unit, two stages beyond
#endif
inline bool fits_128_tiles(long long m, long long n, long long batch, long long cus)
{
    return batch * ((m + 127) / 128) * ((n + 127) / 128) <= A8W8_SMALL_TILES_PER_CU * cus;
}

// Up to 128 activation rows, 128 x 64 tiles instead of 128 x 128: when the wide tiles would occupy at most half of the compute units and the K loop is long
// enough for the deeper staging to matter (a problem of a few K steps is bound by launch and store latency, which narrower tiles
// do not change).
#ifndef A8W8_NARROW_MIN_KSTEPS
#define A8W8_NARROW_MIN_KSTEPS 16
#endif
inline bool narrow_tiles_pay(long long items128, long long n, long long k_bytes, long long cus)
{
    return 2 * items128 <= cus && n > 64 && k_bytes / 128 >= A8W8_NARROW_MIN_KSTEPS;
}

// 256 x 128 tiles where 128 x 128 ones would put two workgroups on a compute unit, 256 x 128 ones would not, and the K loop is
// long enough to make up for a prologue and a tile's stores that no second workgroup hides.  us per launch, bf16 C, two-stage
// 128-tiles -> 256 x 128 (row/col, row-major MX, tiled MX, MXFP4 row-major / tiled, bf16):
//   2560^3            22.2 -> 20.3, 26.1 -> 23.5, 23.3 -> 20.3, 16.8 / 13.9 -> 16.7 / 14.1, 41.3 -> 36.5
//   2049x3584x4096    34.6 -> 28.5, 45.1 -> 36.0, 35.7 -> 30.2, 29.0 / 21.7 -> 24.6 / 19.8, 66.4 -> 51.5
//   512x16384x7168    67.3 -> 57.1, 88.6 -> 81.5, 71.1 -> 60.2, 42.7 / 33.3 -> 39.1 / 29.5, 126.4 -> 112.5
//   2048x4096x2048    18.0 -> 18.1, 21.3 -> 20.2, 19.4 -> 18.6, 15.2 / 12.7 -> 15.8 / 13.5, 31.1 -> 30.1
//   1000x8192x1024    14.2 -> 14.7, 14.9 -> 15.2, 14.3 -> 14.4, 11.8 / 10.7 -> 13.3 / 12.1, 19.1 -> 20.1
// i.e. the line lies at 16 steps of 128 bytes, and where a step's scales cost next to nothing beside its short MFMAs at 24.
constexpr int tall_min_ksteps(bool cheap_steps) { return cheap_steps ? 24 : 16; }

// LDS stages of 128 x 64 tiles: three, or as many as fit 160 KiB (five or six).  Up to 128 rows always those: the workgroup's share of the weights comes from HBM, and a
// deep queue hides its latency (us, three / six, weights from HBM: row-major MX 5 x 3328 x 2688 11.5 / 10.2, 1 x 8064 x 3584 15.4 / 13.8, 13 x 9344 x 2688 12.4 / 11.8,
// MXFP4 2 x 768 x 13312 28.7 / 26.7, 3 x 4736 x 13312 30.0 / 28.7).  The same up to 384 rows for weights that a cache does not keep from one layer's pass to the next, from 12 MiB where a
// step is little more than its operands (STEP_LIGHT: per-tensor, row/col and tiled MXFP8 scales, bf16; whole steps) and from 20 MiB with block scales (from HBM, from the caches: row/col
// 156 x 7936 x 2816 16.1 / 14.7, 13.9 / 13.9, tiled MXFP8 132 x 8064 x 2432 15.2 / 14.4, 13.4 / 13.8; block 186 x 6144 x 7936 34.4 / 30.5, 303 x 4736 x 7680 36.2 / 32.8,
// 177 x 6144 x 5760 26.1 / 23.0, 21.6 / 22.1; not smaller ones, 6 to 12 MiB 1.05 times as long from either, nor other kinds of step: row-major MX 2 to 5% longer, MXFP4 2 to 6%,
// partial steps 4%).  Otherwise beyond 128 rows from 28 light steps on: 1000 x 1536 x 1024 5.9 / 6.3, 402 x 1920 x 3072 10.3 / 10.5, 1024 x 2048 x 4096 13.7 / 13.0, 1495 x 1344 x 7168
// 20.6 / 19.8; tiled MXFP8 11.0 / 11.4 at 24 steps, 14.5 / 14.2 at 32.  Others: block scales 1024 x 2048 x 4096 14.9 / 15.4, row-major MX 20.8 / 22.2, MXFP4 23.5 /
// 24.9, tiled 14.7 / 14.9; partial steps 800 x 2000 x 2000 12.8 / 14.2.
enum StepKind { STEP_LIGHT, STEP_BLOCK, STEP_OTHER };
inline bool narrow_tiles_deep(long long m, long long n, long long k_bytes, StepKind kind)
{
    if (m <= 128 || (kind == STEP_LIGHT && k_bytes / 128 >= 28)) return true;
    return m <= 384 && kind != STEP_OTHER && n * k_bytes >= (kind == STEP_LIGHT ? 12ll << 20 : 20ll << 20);
}

// The variant of the 128-tile kernel: the smallest tile whose workgroups do not outnumber the compute units, since a workgroup alone on its
// compute unit takes as long as its own K loop, and that as long as its tile's rows take from L2 (16, 24, 32 KiB a step: 0.18, 0.27, 0.36 us).
// Beyond 128 activation rows (up to there the flat GEMM's cost model goes by the tiles of narrow_tiles_pay):
//  64 x 64: us, row/col scales, 128 x 128 / 128 x 64 / 64 x 64: 1024 x 1024 x 1024 6.7 / 5.6 / 4.5, 200 x 512 x 512 5.6 / 4.7 / 3.7, 300 x 3072 x 3072
//   12.5 / 10.3 / 7.9, 512 x 2048 x 8192 23.7 / 19.1 / 14.6, bf16 4 x 162 x 384 x 3840 23.9 / 19.4 / 15.1; block scales 1024 x 1024 x 4096 18.1 / 13.8 / 11.1;
//   row-major MX 512 x 512 x 1024 7.4 / 6.3 / 5.0; K = 2000 (a partial step) 1000 x 1000 16.8 / 12.4 / 9.8.  Not for two workgroups per compute unit (700 x
//   2048 x 2048, 352 tiles of 64 x 64 9.7 / 8.3 / 9.2).
//  128 x 64: 1000 x 1536 x 1024 7.3 / 5.9, 1437 x 1280 x 1152 7.6 / 6.4, 1495 x 1344 x 7168 23.3 / 19.8, 512 x 4096 x 1024 on row-major MXFP4 8.9 / 7.5.  Fewer than 16 steps: up
//   to seven eighths of the compute units.  With block scales and fp32 C also where 128 x 128 ones fill more than three quarters of the chip, up to eight steps and from
//   eight columns of them on (block_fp32: two workgroups per compute unit hide each other's multiply-adds and long stores).  128 x 64 / 128 x 128, operands in
//   the caches, from HBM: 2048 x 2048 x 512 8.3 / 8.9, 9.7 / 10.0, x 1024 10.4 / 10.8, 12.4 / 12.2, 8 x 512 x 1024 x 1024 11.6 / 12.3, 3200 x 1024 x 1024 9.5 / 9.6, 11.1 / 11.1,
//   7 x 512 x 1024 x 1024 10.9 / 11.5, 13.4 / 12.4.  Not with bf16 C (2048 x 2048 x 1024 9.0 / 8.6, 11.1 / 9.9), more steps (x 4096 fp32 22.6 / 22.2, 29.4 / 25.4, bf16 21.8 /
//   19.8, 27.2 / 22.5) or fewer columns (16 x 512 x 512 x 4096 46.2 / 33.3, x 1024 15.2 / 13.6, 24640 x 128 x 1024 10.3 / 9.9, 13.5 / 12.2).
// Then, up to one workgroup per compute unit: four LDS stages (deep prefetch).  More: 256 x 128 tiles
// where they pay (has_tall: the variant exists for the operands), else two stages, so that two workgroups share a compute unit and
// hide each other's waits.  cheap_steps: bf16, and MXFP4 on tiled scales.
enum Tile128 { TILES_128x64, TILES_128_FOUR_STAGES, TILES_256x128, TILES_128_TWO_STAGES, TILES_64x64 };
inline Tile128 tile128_variant(long long m, long long n, long long k_bytes, long long batch, bool has_tall, bool cheap_steps, long long cus, bool block_fp32 = false)
{
    const long long tiles_n = (n + 127) / 128, items = batch * ((m + 127) / 128) * tiles_n;
    if (m <= 128) {
        if (narrow_tiles_pay(items, n, k_bytes, cus)) return TILES_128x64;
    } else {
        const long long columns64 = (n + 63) / 64, items64 = batch * ((m + 127) / 128) * columns64;
        if (batch * ((m + 63) / 64) * columns64 <= cus) return TILES_64x64;
        if (8 * items64 <= (k_bytes / 128 >= A8W8_NARROW_MIN_KSTEPS ? 8 : 7) * cus) return TILES_128x64;
        if (block_fp32 && 4 * items > 3 * cus && items <= cus && tiles_n >= 8 && k_bytes <= 8 * 128) return TILES_128x64;
    }
    if (items <= A8W8_SMALL_DEEP_UP_TO * cus) return TILES_128_FOUR_STAGES;
    if (has_tall && batch * ((m + 255) / 256) * tiles_n <= cus && k_bytes / 128 >= tall_min_ksteps(cheap_steps)) return TILES_256x128;
    return TILES_128_TWO_STAGES;
}

// ---------------------------------------------------------------- tiles and XCDs
// Whether an XCD (workgroup ids modulo 8) takes a run of consecutive tiles, which are numbered down eight tile rows and then along the columns, or every eighth
// tile.  The former where 8 divides the tiles.  Elsewhere too up to seven tile rows: a run holds all rows of a few columns, every eighth tile nearly all columns.
// With more rows every eighth tile is one row of the eight, with all columns, and a run of the last, lower group of rows has many more of its columns than the
// other runs have; runs pay where a launch has several tiles per compute unit, so that an XCD's are not all read at once, or many columns and a long K loop.
// us, every eighth tile / runs, tile rows x columns: 128-tile kernel 3 x 52 12.2 / 11.3, 5 x 23 10.6 / 10.0, batch of 8 of 7 x 3 18.0 / 14.9; 17 x 12 12.9 / 13.9,
// 28 x 9 25.2 / 26.3, 42 x 6 29.5 / 31.7, 52 x 7 17.4 / 18.8, 41 x 5 19.0 / 20.8; 25 x 57 63.7 / 55.2, 59 x 13 23.3 / 24.6; 9 x 28 of 55 steps 52.0 / 47.7.  By groups of shapes,
// runs against every eighth tile: fewer than 8 rows 2.5% faster, 9 to 15 rows 2%, 17 and more 4% slower; more than one tile per compute unit and 9 to 15
// rows 1.5% faster, more than two and 21 columns 6%; 40 steps and 13 columns 2% faster.  A batch of two or four rows of tall tiles (128 x 64, 256 x 128) shares a tile row's
// A, the larger operand, among every eighth tile: 16 of 2 x 6 12.0 / 12.9, 20.5 / 22.7, 16 of 4 x 3 42.1 / 46.6, 8 of 4 x 7 51.1 / 70.9.
inline bool tiles_in_runs(long long tiles_m, long long tiles_n, long long k_steps, long long batch, bool tall, long long cus)
{
    const long long tiles = tiles_m * tiles_n;
    if (tiles % 8 == 0) return true;
    if (tiles_m < 8) return !(batch > 1 && 8 % tiles_m == 0 && tall);
    return (tiles > cus && tiles_m < 16) || (tiles > 2 * cus && tiles_n > 20) || (k_steps >= 40 && tiles_n > 12);
}
// The same for the 256-tile kernels, whose workgroups walk the tiles of all batch entries: up to two rounds of them and fewer than 16 steps runs are 2% slower (9 x 28 31.4 /
// 33.4, 9 x 21 19.9 / 21.4), longer or more rounds 1 to 4% faster (220 tiles of 40 steps 59.0 / 58.0, 26 x 31 of 38 steps 300 / 281).
inline bool items_in_runs(long long tiles_m, long long tiles_n, long long k_steps, long long batch, long long cus)
{
    const long long tiles = tiles_m * tiles_n;
    return tiles % 8 == 0 || tiles_m < 8 || k_steps >= 16 || batch * tiles > 2 * cus;
}

// ---------------------------------------------------------------- flat GEMM (up to 128 activation rows)
// Weight tiles (nt) and groups of 16 activation rows (mt) per workgroup of the flat GEMM.
//
// Below four weight tiles per compute unit: the smallest nt x mt whose workgroups all fit the chip at once.  Every workgroup is
// eight waves and a chain of K pairs, reduction and store whose length grows with nt x mt, so a layer of few weight tiles goes out in
// small pieces (row groups then read the weights once each, all but the first from L2), and one of many in pieces large enough for
// a single round.  us, row/col / MXFP8, fixed splits -> these:
//   64 x 1024 x 4096     2 x 4  8.7 / 9.9   -> 1 x 1  5.2 / 6.1       100 x 1024 x 4096   2 x 8, 2 x 4  13.2 / 9.8 -> 1 x 2  5.2 / 6.0
//   64 x 4096 x 4096     2 x 4  9.2 / 10.5  -> 2 x 2  7.1 / 8.0       100 x 4096 x 4096   2 x 8, 2 x 4  14.2 / 10.6 -> 2 x 4  9.3 / 10.6
//   64 x 9216 x 3584     2 x 4  14.6 / 17.8 -> 4 x 4  12.8 / 13.1     128 x 8192 x 8192   2 x 8, 2 x 4  25.9 / 33.4 -> 4 x 4  23.3 / 24.2
//   128 x 12288 x 2560   2 x 8  20.7 -> 2 x 4 in three rounds 16.2 (MXFP8: 2 x 4 17.9 before and now, 4 x 4 19.0)
//   16 x 5120 x 5120     1 x 1  9.9 / 11.4  -> 2 x 1  8.0 / 8.7       16 x 10240 x 8192   2 x 1  19.9 / 22.5 -> 4 x 1  17.4 / 18.6
// Four row groups share a pass at most, six where their registers allow it (MX scales: only over a few K pairs; otherwise 4 x 4 on two
// passes is faster, 80 x 7168 x 4096 14.6 -> 13.4).
//
// Two weight tiles stay two, in up to two rounds, where four would make the chain longer than they save:
//  - rows of at most 1024 bytes (MX formats 512), one K pair or less per wave: four tiles only lengthen reduction and stores
//    (four / two tiles: 32 x 14336 x 1024 6.1 / 5.5, block scales 48 x 14336 x 1024 7.4 / 6.7, MXFP4 64 x 12288 x 1024 6.1 / 5.8).  Not
//    where a workgroup stages row-major weights beside three or four row groups (tensor 64 x 10240 x 512 two tiles 29% slower), nor
//    for block scales with four groups (64 x 12288 x 512 18% slower), nor for nine to sixteen rows over rows of more than 512 bytes
//    and less than 3.25 tiles per compute unit (16 x 10240 x 1024 4% slower);
//  - up to eight activation rows over at least 3.25 tiles per compute unit, where two rounds of two tiles are nearly full and there
//    are few activation bytes to share (four / two: 1 x 14336 x 8192 20.1 / 18.9, bf16 1 x 15360 x 4096 22.0 / 20.5); on row-major weights,
//    whose rows a workgroup stages through LDS, for rows of up to 2048 bytes, without MX scales from two tiles on (1 x 12288 x 2048
//    7.6 / 7.2, 16 x 15360 x 2048 8.8 / 8.4; beyond 2048 bytes four are 8 to 11% faster: bf16 8 x 13312 x 8192).
// One tile stays one for up to four rows over row-major weights with per-tensor, row/col or no scales and rows of up to 8192 bytes
// (two / one: 1 x 7168 x 8192 11.7 / 10.7, bf16 1 x 6144 x 4096 11.1 / 10.4; bf16 4 x 6144 x 8192 the other way, 8%).
//
// Layers of at least four weight tiles per compute unit take four, and an even split of the row groups over one or two passes (16384 x
// 7168 at M = 48, 30 us with two tiles, 24 us with four).
enum FlatKind { FLAT_FP8, FLAT_BLOCK, FLAT_BF16, FLAT_MXFP8, FLAT_MXFP4 };      // (FLAT_FP8: per-tensor and row/col scales)
struct FlatSplit { int nt, mt; };
inline FlatSplit flat_split(FlatKind kind, bool row_major, long long m, long long n, long long row_bytes, long long batch, long long cus)
{
    const bool mx = kind == FLAT_MXFP8 || kind == FLAT_MXFP4;
    const long long tiles = n / 16 * batch;
    const int groups = (int)((m + 15) / 16), passes = (groups + 3) / 4, mt = (groups + passes - 1) / passes;
    if (tiles >= 4 * cus) return {4, mt};
    const auto fits = [&](int nt, int g) { return (n / 16 + nt - 1) / nt * batch * ((groups + g - 1) / g) <= cus; };
    const bool short_rows = row_bytes <= (mx ? 512 : 1024);
    if (fits(1, 1)) return {1, 1};
    if (groups == 1) {
        if (fits(2, 1)) return row_major && (kind == FLAT_FP8 || kind == FLAT_BF16) && m <= 4 && row_bytes <= 8192 ? FlatSplit{1, 1} : FlatSplit{2, 1};
        const bool full = 4 * tiles >= 13 * cus, two_rounds_full = m <= 8 && full;
        if (m > 8 && !full && row_bytes > 512) return {4, 1};
        return short_rows || (row_major ? row_bytes <= 2048 && (!mx || two_rounds_full) : two_rounds_full) ? FlatSplit{2, 1} : FlatSplit{4, 1};
    }
    if (fits(1, 2)) return {1, 2};
    if (fits(2, 2)) return {2, 2};
    if (groups > 2 && fits(2, 3)) return {2, 3};
    if (groups > 2 && fits(2, 4)) return {2, 4};
    if (groups <= 4) return {short_rows && (groups == 2 || (!row_major && !(kind == FLAT_BLOCK && groups == 4))) ? 2 : 4, mt};
    if (groups <= 6) return !mx || short_rows ? FlatSplit{2, 6} : FlatSplit{4, 4};
    if (!fits(4, 4) || (kind == FLAT_MXFP4 && !row_major && short_rows)) return {2, 4};
    return {4, 4};
}

// The flat GEMM against the 128-tile kernel on problems of at most 128 activation rows: true where this cost model calls the flat one
// faster.  Times in microseconds, W = weight bytes, row_bytes = bytes of one weight row:
//   flat:  one pass over the weights at ~6.4 TB/s; every further group of 16 activation rows adds the activation rows
//          that each workgroup reads again for its weight tiles, W / NT bytes at ~21 TB/s (1.4 us on 16384 x 7168), nearly twice
//          that where the workgroups do not fit the chip at once; a second pass (more than 64 rows over at least four weight
//          tiles per compute unit) reads the weights from L2 and costs 55% more; MXFP8 a tenth (layout_factor).
//   dense: the 128-tile kernel pulls the weights with one workgroup per 128 weight rows at ~28 GB/s each, or, where
//          128 x 128 tiles would occupy at most half of the compute units, per 64 rows at ~22 GB/s each (its 128 x 64
//          tiles), ~5 TB/s at best over the chip; 20% more at 128 activation rows than at a few.
// Weights of at most 32 MiB (per batch entry) always go flat.  Measured, shuffled FP8 weights, M = 16 / 32 / 48 / 64 / 80 / 96 / 128, flat
// against dense:
//   16384 x 7168   20 / 21 / 23 / 24 / 35 / 36 / 41  against  30 / 27 / 27 / 28 / 30 / 31 / 33   (MXFP8 about 10% more on both sides)
//   8192 x 8192    13 / 14 / 16 / 18 / 21 / 22 / 23  against  26 / 26 / 26 / 27 / 28 / 29 / 31
//   28672 x 4096   20 / 23 / 25 / 28 / 39 / 41 / 47  against  26 / 26 / 27 / 28 / 29 / 30 / 31
//   4096 x 14336   13 / .. / .. / 19 / 23 / .. / 27  against  41 throughout
// (tests/test_zz_gpu_routing.py times both sides of such cells through a8w8_route_override and checks the choice).  Over 3936 cells (six kinds
// of operands, both layouts, M = 16 .. 128, 2048 .. 28672 columns, batches of 1, 2 and 4) the choice costs 1.0% over the better
// side in the mean and is more than 10% off in 4% of them.
// NT here is what the fit was made with, not what flat_split takes today: four for one to four groups past two tiles per compute
// unit, but two for five to eight groups there, whose 2 x 6 or 4 x 4 on two passes costs per group as two tiles do (four in the
// formula: 17% of the cells more than 10% off).
// The batch: more than four groups are priced over all entries together (128 x 8192 x 8192 MXFP8, four entries: flat 99, dense 66).  Up to
// four are priced by the entry, which is within 5% except between two and four tiles per compute unit on more than 128 MiB of weights
// in all (64 x 14336 x 14336, two entries: flat 88, dense 78; 64 x 14336 x 4096, two: 28, 31): two tiles there, as for large grids.
inline bool flat_is_faster(long long m, long long n, long long row_bytes, long long batch, double layout_factor, long long cus)
{
    const double w_entry = (double)n * (double)row_bytes;
    if (w_entry <= (double)(32ll << 20)) return true;
    const int groups = (int)((m + 15) / 16), passes = (groups + 3) / 4, mt = (groups + passes - 1) / passes;
    const long long entries = groups > 4 ? std::max(batch, 1ll) : 1;
    const double w = w_entry * (double)entries;
    const long long tiles = n / 16 * entries, tiles128 = (n + 127) / 128 * entries;
    const bool small_batch = batch <= 1 || w_entry * (double)batch <= (double)(128ll << 20);
    const int nt = tiles >= 4 * cus || (groups <= 4 && tiles > 2 * cus && small_batch) ? 4 : tiles > cus ? 2 : 1;
    const double per_group = w / nt / 21.0e6 * (tiles / nt > cus ? 1.9 : 1.0);
    double flat = 1.5 + w / 6.4e6;
    if (groups > 4 && tiles < 4 * cus) {
        flat += per_group * (groups - 1);      // six row groups in one pass, or two passes of workgroups of four (see flat_split)
    } else {
        flat += per_group * (mt - 1);
        if (passes == 2) flat *= 1.55;         // the second pass reads the weights from L2
    }
    flat *= layout_factor;      // row-major weights: rows staged through LDS, rows a power of two apart share channels
    // (the 128-tile kernel's own choice of tile width for one row of 128-row tiles)
    const bool narrow = narrow_tiles_pay(tiles128, n, row_bytes, cus);
    const long long rounds = (tiles128 + cus - 1) / cus;
    const double per_workgroup = narrow ? 64.0 * (double)row_bytes / 22.0e3 : (double)rounds * 128.0 * (double)row_bytes / 28.0e3;
    double dense = 4.0 + std::max(per_workgroup, w / 5.0e6);
    dense *= 1.0 + 0.2 * (double)m / 128.0;
    return flat <= dense;
}

}  // namespace a8w8
