// Which kernel variant a call takes, where that depends on its sizes: plain host functions of sizes and the number of compute
// units, without the HIP runtime, so that they can be checked without a GPU.  Times in the comments: MI355X, 256 compute units,
// us per launch inside a graph.
#pragma once

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
inline bool f4_row_scales_on_256_tiles(long long m, long long n, long long k_steps, long long batch, bool fp32_c, long long cus)
{
    const long long rounds128 = (batch * ((m + 127) / 128) * ((n + 127) / 128) + cus - 1) / cus;
    const long long rounds256 = (batch * ((m + 255) / 256) * ((n + 255) / 256) + cus - 1) / cus;
    if (k_steps < (fp32_c ? 8 : 4)) return false;
    return 2 * rounds128 >= (k_steps >= (fp32_c ? 16 : 12) ? 6 : 7) * rounds256;
}

}  // namespace a8w8
