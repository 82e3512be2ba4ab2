// What the dense A8W8 GEMM kernels for gfx950 share: the 256 x 256 x 128 workgroup tile of the
// pipelined kernels (gemm_persist.hpp: 8 waves, 64 x 128 per wave; gemm_wide.hpp: 4 waves,
// 128 x 128 per wave), its LDS budget, and the workgroup-id -> tile mapping.
//
// Data path of every kernel: A and B tiles go global -> LDS with 16-byte direct-to-LDS buffer
// loads into 128-byte LDS rows (one K step of one matrix row) whose 16-byte slots are
// XOR-swizzled on the global-address side (the direct-to-LDS write itself is always
// wave-linear) and un-swizzled by the readers, which keeps the 64-lane ds_read_b128 free of
// bank conflicts.
//
// MFMA operand roles are swapped with respect to the matrix names: rows of B (index n)
// feed the MFMA "A" operand and rows of A (index m) the "B" operand, so that a lane ends
// up holding C[m = lane%16][n = 4*(lane/16) .. +3]: four consecutive n, one 8-byte store
// of bf16, and one A-side scale per lane per tile.
#pragma once
#include <type_traits>
#include <utility>

#include "a8w8_device.hpp"

namespace a8w8 {

constexpr int BM = 256, BN = 256, BK = 128;
constexpr int GEMM_THREADS = 512;
constexpr int STAGE_BYTES = (BM + BN) * BK;          // 65536
constexpr int GEMM_LDS_BYTES = 2 * STAGE_BYTES;      // 131072
// MX only: E8M0 scales of 4 K steps (16 bytes per row, 256 A rows then 256 B rows), two buffers
constexpr int MX_GROUP_BYTES = (BM + BN) * 16;       // 8192
constexpr int GEMM_LDS_BYTES_MX = GEMM_LDS_BYTES + 2 * MX_GROUP_BYTES;
constexpr int WAVE_M = 64, WAVE_N = 128;
constexpr int TM = WAVE_M / 16, TN = WAVE_N / 16;    // 4 x 8 MFMA tiles per wave

// Workgroup id -> tile (tile_of_block).  Consecutive workgroup ids land on different XCDs (round-robin over
// 8), each with its own L2, so ids are first regrouped so that one XCD works on a
// contiguous run of tiles, except on some tile counts that 8 does not divide (`runs`: tiles_in_runs and items_in_runs of routes.hpp); inside the run, tiles are
// walked down 8 tile-rows before moving to the next tile-column so that concurrently resident tiles share A rows and B rows.
// Nothing hides the lookup (the persistent kernels look tiles up at every tile change, the 128-tile kernel in front of its first load): every division is by a value the host knows, so the host passes floor(2^32 / d) for each of them and the
// kernel divides with one multiply and one correction (exact for 0 <= n < 2^31 and any d >= 1: the estimate
// mulhi(n, floor(2^32 / d)) is the quotient or one less).  Measured against run-time divisors: 0.25% of the MXFP8 8192^3
// launch (four tiles per workgroup), 1-2% of block-scale 4096 x 7168 x 2048 (two tiles of 16 K steps).
struct TileMap {
    int tiles_m, tiles_n;
    int tiles;                 // tiles_m * tiles_n
    int per_group;             // 8 * tiles_n: the tiles of eight tile rows
    int rem;                   // tiles_m % 8: tile rows of the last group when it is not a full one (0: none)
    uint32_t inv_tiles, inv_per_group, inv_rem;      // floor(2^32 / d) of the three divisors (d = 1: 2^32 - 1)
    int runs;                  // a run of tiles per XCD
};
__host__ __device__ inline uint32_t tile_map_inverse(int d)
{
    return d <= 1 ? 0xFFFFFFFFu : (uint32_t)((1ull << 32) / (uint32_t)d);
}
__host__ inline TileMap make_tile_map(int tiles_m, int tiles_n, bool runs)
{
    TileMap t;
    t.tiles_m = tiles_m; t.tiles_n = tiles_n;
    t.tiles = tiles_m * tiles_n;
    t.per_group = 8 * tiles_n;
    t.rem = tiles_m % 8;
    t.inv_tiles = tile_map_inverse(t.tiles);
    t.inv_per_group = tile_map_inverse(t.per_group);
    t.inv_rem = tile_map_inverse(t.rem);
    t.runs = runs;
    return t;
}
A8W8_DEV int div_by_known(int n, int d, uint32_t inv)
{
    int q = (int)__umulhi((uint32_t)n, inv);
    if (n - q * d >= d) ++q;
    return q;
}
A8W8_DEV void tile_of_block(const GemmParams& p, int bid, int& tm, int& tn)
{
    const int nt = p.tiles_m * p.tiles_n;
    // (runs of nt / 8 tiles, the first nt % 8 of them one longer)
    const int id = p.runs ? (bid & 7) * (nt >> 3) + min(bid & 7, nt & 7) + (bid >> 3) : bid;
    const int per_group = 8 * p.tiles_n, group = div_by_known(id, per_group, p.inv_per_group), first_m = group * 8, in_group = id - group * per_group;
    if (p.tiles_m - first_m >= 8) {
        tn = in_group >> 3;
        tm = first_m + (in_group & 7);
    } else {
        const int rem = p.tiles_m & 7;
        tn = div_by_known(in_group, rem, p.inv_rem);
        tm = first_m + in_group - tn * rem;
    }
}
// work item (batch entry, tile) -> batch entry and tile coordinates
A8W8_DEV void tile_of_item(const TileMap& t, int item, int& batch, int& tm, int& tn)
{
    batch = div_by_known(item, t.tiles, t.inv_tiles);
    const int bid = item - batch * t.tiles;
    const int id = t.runs ? (bid & 7) * (t.tiles >> 3) + min(bid & 7, t.tiles & 7) + (bid >> 3) : bid;
    const int group = div_by_known(id, t.per_group, t.inv_per_group);
    const int first_m = group * 8;
    const int in_group = id - group * t.per_group;
    if (t.tiles_m - first_m >= 8) {
        tn = in_group >> 3;
        tm = first_m + (in_group & 7);
    } else {
        tn = div_by_known(in_group, t.rem, t.inv_rem);
        tm = first_m + in_group - tn * t.rem;
    }
}

// Accumulators in named registers, for the kernels with one wave per SIMD: the four-wave kernel's 64 tiles (i, j) of a wave
// live in accumulator registers a[4 (8i + j) : +3], the 32 of the 256 x 128 variant of the 128-tile kernel in a[4 (4i + j) : +3].
// (Left to the compiler, a loop of 32 tiles moved every accumulator through one register quadruple, with the idle cycles between
// an MFMA and the read of its result each time: twice the time per K step.)  They are named in assembly statements only and never appear as variables: the
// compiler allocates nothing there (its own registers stay below 256, which the build checks), so no
// copy, spill or re-materialisation can come between two MFMAs of one tile.  The statements keep
// their order; the compiler does not see the MFMAs' latency, so the code that reads an accumulator
// makes sure that enough instructions separate it from the last MFMA into that tile.
template <int N, class F, int... I>
A8W8_DEV void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
A8W8_DEV void static_for(F&& f)
{
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// tile LO/4 += a . b, or = a . b when ZC (the tile's first K step)
template <int LO, bool ZC>
A8W8_DEV void mfma_acc(const v8i& a, const v8i& b)
{
    if constexpr (ZC) asm volatile("v_mfma_f32_16x16x128_f8f6f4 a[%2:%3], %0, %1, 0" ::"v"(a), "v"(b), "n"(LO), "n"(LO + 3));
    else asm volatile("v_mfma_f32_16x16x128_f8f6f4 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(LO), "n"(LO + 3));
}
// the same with E8M0 block scales: byte OA of sa scales a's K block of the lane, byte OB of sb b's
template <int LO, bool ZC, int OA, int OB>
A8W8_DEV void mfma_acc_mx(const v8i& a, const v8i& b, int sa, int sb)
{
    if constexpr (ZC)
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[%4:%5], %0, %1, 0, %2, %3 op_sel:[%6,%7,0] op_sel_hi:[%8,%9,0]" ::"v"(a),
                     "v"(b), "v"(sa), "v"(sb), "n"(LO), "n"(LO + 3), "n"(OA & 1), "n"(OB & 1), "n"(OA >> 1), "n"(OB >> 1));
    else
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[%4:%5], %0, %1, a[%4:%5], %2, %3 op_sel:[%6,%7,0] op_sel_hi:[%8,%9,0]" ::"v"(a),
                     "v"(b), "v"(sa), "v"(sb), "n"(LO), "n"(LO + 3), "n"(OA & 1), "n"(OB & 1), "n"(OA >> 1), "n"(OB >> 1));
}
// bf16 operands: one 16 x 16 x 32 MFMA per 16-byte half of a fragment
template <int LO, bool ZC>
A8W8_DEV void mfma_acc_bf16(const v4i& a, const v4i& b)
{
    if constexpr (ZC) asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, 0" ::"v"(a), "v"(b), "n"(LO), "n"(LO + 3));
    else asm volatile("v_mfma_f32_16x16x32_bf16 a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(LO), "n"(LO + 3));
}
// packed E2M1 operands (format 4 for both): one 16 x 16 x 128 MFMA per 16-byte half of a fragment
template <int LO, bool ZC, int OA, int OB>
A8W8_DEV void mfma_acc_f4(const v4i& a, const v4i& b, int sa, int sb)
{
    if constexpr (ZC)
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[%4:%5], %0, %1, 0, %2, %3 op_sel:[%6,%7,0] op_sel_hi:[%8,%9,0] cbsz:4 blgp:4" ::"v"(a),
                     "v"(b), "v"(sa), "v"(sb), "n"(LO), "n"(LO + 3), "n"(OA & 1), "n"(OB & 1), "n"(OA >> 1), "n"(OB >> 1));
    else
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[%4:%5], %0, %1, a[%4:%5], %2, %3 op_sel:[%6,%7,0] op_sel_hi:[%8,%9,0] cbsz:4 blgp:4" ::"v"(a),
                     "v"(b), "v"(sa), "v"(sb), "n"(LO), "n"(LO + 3), "n"(OA & 1), "n"(OB & 1), "n"(OA >> 1), "n"(OB >> 1));
}
template <int IDX>
A8W8_DEV float acc_read()
{
    float x;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(IDX));
    return x;
}

template <int IDX>
A8W8_DEV void acc_zero()
{
    asm volatile("v_accvgpr_write_b32 a[%0], 0" ::"n"(IDX));
}

}  // namespace a8w8
