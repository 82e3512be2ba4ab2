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

}  // namespace a8w8
