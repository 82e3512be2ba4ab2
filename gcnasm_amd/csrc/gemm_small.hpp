// Dense GEMM for problems too small to fill the chip with 256 x 256 tiles: 128 x 128 x 128 tile, 4 waves
// (2 along M x 2 along N), each wave owning a 64 x 64 block of C as 4 x 4 MFMA tiles of 16 x 16 x 128.
// A quarter of the work per workgroup means four times as many workgroups, and a problem of this size is
// bound by latency (first loads, the K loop's dependent steps, the C stores of one compute unit), not by the
// matrix cores.
//
// Data path as in the 256-tile kernels: 16-byte direct-to-LDS loads, 128-byte LDS rows whose 16-byte slots are
// XOR-swizzled with (row & 7), operand roles swapped so that a lane ends up with
// C[m = lane%16][n = 4*(lane/16) .. +3].  LDS stages of 32 KiB, four (loads three K steps ahead, one raw
// barrier per step) or two (see the kernel's template parameter).  Scales that change with the K step -- block
// scales, MX exponents -- ride in the same pipeline: each stage carries its step's scales, fetched by one extra
// direct-to-LDS load per wave, so that the loop's wait counts stay fixed and no global load has to be waited
// for inside a step.  Operands: FP8 E4M3, bf16 (byte rows of 2k columns), packed E2M1 (byte rows of k/2 columns).
#pragma once
#include "gemm_common.hpp"

namespace a8w8 {

constexpr int SM_BM = 128, SM_BN = 128;               // the usual tile; the kernel also takes 64 columns, 64 x 64, or 256 rows
constexpr int SM_THREADS = 256;
constexpr int small_stage_bytes(int bn, int bm = SM_BM) { return (bm + bn) * BK; }   // 128 x 128: 32768, 128 x 64: 24576, 256 x 128: 49152
// Scale bytes per stage.  Block mode: 128 A-row scales, the B scale at +512 and +768.  Row-major MX: the step's
// four E8M0 bytes of 128 A rows, then of 128 B rows.  Tiled MX: 1 KiB per wave, whose first half is the 512-byte
// unit (64 rows x one pair of K steps) of the wave's row block.
// Row-major MX scales of packed E2M1 operands (MODE_F4): a 128-byte K step is 256 elements, eight E8M0 bytes per row:
// the rows' first dwords (128 A rows, then 128 B rows), then their second dwords.
// 256-row tiles: row-major MX 256 A rows, then the 128 B rows (twice); MODE_F4 the same with A's second dwords behind A's first
// and B's behind B's; tiled MX the six 512-byte units of the tile (four A blocks, two B blocks), two per wave.
constexpr int small_scale_bytes(int mode, int bm = SM_BM)
{
    if (bm == 256) return mode == MODE_MX ? 2048 : mode == MODE_MXT || mode == MODE_F4T || mode == MODE_F4 ? 4096 : 0;
    return mode == MODE_MXT || mode == MODE_F4T ? 4096 : mode == MODE_F4 ? 2048 : (mode == MODE_BLOCK || mode == MODE_MX) ? 1024 : 0;
}
#ifndef A8W8_SMALL_PIPELINED
#define A8W8_SMALL_PIPELINED 1          // 0: loads in a block behind the barrier, fragments read in their own step (measurement)
#endif
#ifndef A8W8_SMALL_PIPELINED_TWO
#define A8W8_SMALL_PIPELINED_TWO 1      // the same switch for the two-stage variant
#endif
#ifndef A8W8_SMALL_LINES_BY_LANE
#define A8W8_SMALL_LINES_BY_LANE 1      // 0: whole tiles are stored from the MFMA layout as they are (measurement)
#endif
constexpr int small_lds_bytes(int mode, int stages, int bn = SM_BN, int bm = SM_BM)
{
    return stages * (small_stage_bytes(bn, bm) + small_scale_bytes(mode, bm)) + (mode == MODE_ROWCOL ? (bm + bn) * 4 : 0);
}

// p.tiles_m / p.tiles_n count 128 x 128 tiles here; grid = (tiles, 1, batch).  The launch bound asks for a
// 256-register budget: with 512 the compiler parks the block mode's partial tiles in accumulation registers
// and copies each value back before its multiply-add.
// SM_STAGES = 4: loads three K steps ahead, one barrier per step, one workgroup per compute unit (132-144 KiB of
// LDS) -- for grids of at most one workgroup per compute unit, where nothing else hides the load latency.
// SM_STAGES = 2: loads issued when a stage has been read, two barriers per step, two workgroups per compute unit
// that hide each other's waits -- for larger grids.
// BN_ = 64: tiles of 128 x 64 (a wave owns 64 x 32) for short, wide problems -- M of a few hundred rows over weights
// of many megabytes -- where 128 x 128 tiles would leave half of the compute units without a workgroup.  A workgroup
// alone on its compute unit streams its share of the weights through a long K loop: SM_STAGES = 6 there (five K
// steps of loads ahead, 144-154 KiB of LDS; 5 with tiled MX scales, whose 4 KiB per stage would not fit six; measured,
// five and six stages run alike, and so does a separate ring of ten stages for the weights); three where steps are few or
// more than their operands (narrow_tiles_deep).
// BM_ = 64: tiles of 64 x 64 (a wave owns 32 x 32), four stages of 16 KiB, for problems of at most one of them per compute unit, where the time
// is one workgroup's K loop: half the operand bytes of a 128 x 64 tile per step (bound: L2 -> LDS, about 90 GB/s per compute unit at any tile size;
// 1024 x 1024 x 1024 5.6 -> 4.5 us, 512 x 2048 x 8192 19.1 -> 14.6).  Splitting K over workgroups instead costs 2.5 to 9 us for the exchange of
// the partial tiles (134 x 1984 x 6912: 16.1 unsplit, 13.4 in three parts, 12.7 on 64 x 64 tiles; 256 x 4096 x 4096 11.5, 13.7, 9.0).
// RAGGED: k is no multiple of 128 (bytes).  The last K step is a partial one: the 16-byte pieces past k are fetched with a
// lane offset beyond the buffer descriptor and read as zero on both sides (k % 16 == 0, so a piece is never split).  FP8
// operands then run on the bf16 MFMA: the one-thread-per-element kernel that took these shapes before adds products in
// fp32 one after the other, and the FP8 MFMA, which aligns its products to the largest one, is about 40 times less
// precise than that (1.4e-5 against 8e-8 of the result in norm over K = 4096 normal data), while E4M3 -> bf16 is exact
// and the bf16 MFMA keeps fp32 sums (8e-8).  A K step is four quarters of 32 elements; the fragments of the next quarter,
// behind the last one those of the next step's first, are converted two instructions per MFMA (in bursts, with the first
// quarter in front of the step's MFMAs: 1024 x 3072 x 2000 19.6 us, 16.9 this way).  Half the MFMA rate, and still bound by it.
// 1000 x 3000 x 2000 row/col: 7545 us on the one-thread-per-element kernel, 18.5 us here; 4096 x 4096 x 4080: 1.2 PFLOP/s.
// BM_ = 256: 256 x 128 tiles, a wave owns 128 x 64 (accumulators in named accumulation registers, one wave per SIMD, three stages
// of 48 KiB), for grids that would need two workgroups per compute unit on 128 x 128 tiles but fit at one per compute unit here.
// A 64 x 64 wave tile reads 16 KiB of LDS per 16 MFMAs and the loads write another 8: as many cycles as the MFMAs take, so
// two workgroups on a compute unit queue for LDS.  128 x 64 reads 24 KiB per 32 MFMAs.  Not for block scales: their
// multiply-adds need the accumulators where the VALU can read them, which 128 of them beside 192 fragment registers are not.
template <int MODE, int CDT, int SM_STAGES, int BN_ = SM_BN, bool RAGGED = false, int BM_ = 128>
__global__ void __launch_bounds__(SM_THREADS, BM_ == 256 ? 1 : 2) __attribute__((amdgpu_waves_per_eu(BM_ == 256 ? 1 : 2, BM_ == 256 ? 1 : 8))) gemm_a8w8_tile128(GemmParams p)
{
    constexpr bool TALL = BM_ == 256;
    constexpr bool SHORT = BM_ == 64;
    static_assert(BM_ == 128 || (SHORT && BN_ == 64 && SM_STAGES > 2) || (TALL && SM_STAGES == 3 && BN_ == 128 && !RAGGED && MODE != MODE_BLOCK), "tile height");
    static_assert(!RAGGED || MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_BF16, "partial K steps: no scales that change with K");
    constexpr bool BY_BF16 = RAGGED && MODE != MODE_BF16;      // FP8 operands converted to bf16
    static_assert(SM_STAGES == 2 || SM_STAGES == 3 || SM_STAGES == 4 || SM_STAGES == 5 || SM_STAGES == 6, "LDS stages");
    static_assert(BN_ == 128 || BN_ == 64, "tile width");
    constexpr int SM_BN = BN_;
    constexpr int SM_BM = BM_;
    constexpr int SM_STAGE_BYTES = small_stage_bytes(SM_BN, SM_BM);
    constexpr int SM_TM = SM_BM / 32;                  // MFMA tiles per wave along M
    constexpr int A_LOADS = SM_BM / 32;                // 1 KiB chunks of A per wave and stage
    constexpr int SM_TN = SM_BN / 32;                  // MFMA tiles per wave along N
    constexpr int B_LOADS = SM_BN / 32;                // 1 KiB chunks of B per wave and stage
    static_assert(MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_BLOCK || MODE == MODE_MX || MODE == MODE_MXT ||
                      MODE == MODE_BF16 || MODE == MODE_F4T || MODE == MODE_F4,
                  "fp32 scales, MX scales, bf16 operands (byte rows of 2k columns, no scales) or packed E2M1 operands (byte "
                  "rows of k/2 columns) with tiled MX scales");
    // tiled scales: of FP8 operands (a K step is 4 blocks of 32: one step of a pair) or of FP4 operands (8 blocks: a pair)
    constexpr bool TILED_SCALES = MODE == MODE_MXT || MODE == MODE_F4T;
    constexpr bool STEP_SCALES = MODE == MODE_BLOCK || MODE == MODE_MX || MODE == MODE_F4 || TILED_SCALES;      // scales that change with the K step
    constexpr bool IS_F4 = MODE == MODE_F4T || MODE == MODE_F4;      // packed E2M1 operands
    constexpr int SM_SCALE_BYTES = small_scale_bytes(MODE, SM_BM);
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = wave_uniform(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1;
    const int batch = blockIdx.z;
    const int r16 = lane & 15, g = lane >> 4;

    // What the first loads' addresses need of the arguments is fetched here, with the tile counts: fetched where it is used, it is a second wait for
    // the argument block in front of the first load.
    asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.sfa), "s"(p.sfb), "s"(p.m), "s"(p.n), "s"(p.k), "s"(p.lda), "s"(p.ldb), "s"(p.a_batch), "s"(p.b_batch),
                 "s"(p.sfa_batch), "s"(p.sfb_batch), "s"(p.stride_sfa), "s"(p.stride_sfb), "s"(p.b_kshift));
    int tile_m, tile_n;
    tile_of_block(p, blockIdx.x, tile_m, tile_n);
    const int m0 = tile_m * SM_BM, n0 = tile_n * SM_BN;
    const int nk = RAGGED ? (p.k + BK - 1) / BK : p.k / BK;

    const uint8_t* a_base = p.a + (long long)batch * p.a_batch;
    const uint8_t* b_base = p.b + (long long)batch * p.b_batch;
    const float* sfa_f = (const float*)p.sfa + (long long)batch * p.sfa_batch;
    const float* sfb_f = (const float*)p.sfb + (long long)batch * p.sfb_batch;
    const __amdgpu_buffer_rsrc_t rsrc_a = make_rsrc(a_base, (uint32_t)(p.m - 1) * p.lda + p.k);
    const __amdgpu_buffer_rsrc_t rsrc_b = make_rsrc(b_base, b_extent_bytes(p));

    // ---- global -> LDS.  A stage holds 16 (or 32) A chunks then 16 (or 8) B chunks of 1 KiB (8 rows x 128 B); wave w
    // fills chunks w, w+4, .. of each matrix.  Lane i of a load lands on row i/8, slot i%8 of its
    // chunk and therefore fetches K-piece slot ^ (row & 7) = (i%8) ^ (i/8).
    const int ld_row = wave * 8 + (lane >> 3);
    const int ld_piece16 = ((lane & 7) ^ (lane >> 3)) * 16;
    // (256-row tiles: one lane offset per operand, the 32 j rows are scalar; rows past the end read as zero or as another
    // row inside the descriptor and only reach accumulators that are never stored)
    int voff_a[TALL ? 1 : A_LOADS], voff_b[TALL ? 1 : B_LOADS];
    if constexpr (TALL) {
        voff_a[0] = (m0 + ld_row) * p.lda + ld_piece16;
        voff_b[0] = b_lane_offset(p, n0 + ld_row, ld_piece16);
    } else {
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) voff_a[j] = min(m0 + ld_row + 32 * j, p.m - 1) * p.lda + ld_piece16;
#pragma unroll
        for (int j = 0; j < B_LOADS; ++j) voff_b[j] = b_lane_offset(p, min(n0 + ld_row + 32 * j, p.n - 1), ld_piece16);
    }
    // the lane's piece of the last, partial K step lies past k: out of every descriptor's range (an extent is below 2^31; 2^31 in
    // place of the lane's offset, not on top of it: together with the scalar offset that could pass 2^32, and wrap into the matrix)
    const bool past_k = RAGGED && (nk - 1) * BK + ld_piece16 >= p.k;
    auto lane_offset = [&](int voff, int kstep) __attribute__((always_inline)) { return RAGGED && past_k && kstep == nk - 1 ? (int)0x80000000u : voff; };
    // block mode: waves 0 and 1 fetch the step's 128 A-row scales (64 each), waves 2 and 3 the B scale
    // of the tile's 128 x 128 block (every lane the same dword: the stage's copy at +512 is the one read)
    constexpr int SF_LOADS = !STEP_SCALES ? 0 : TALL && !TILED_SCALES ? (MODE == MODE_F4 ? 4 : 2) : MODE == MODE_F4 ? 2 : 1;
    constexpr int LOADS_PER_STAGE = A_LOADS + B_LOADS + SF_LOADS;
    __amdgpu_buffer_rsrc_t rsrc_sf = rsrc_a, rsrc_sf_b = rsrc_a;      // (the second one: 256-row tiles, B's scales)
    int voff_sf = 0, voff_sf_b = 0, sf_step_bytes = 0;
    if constexpr (MODE == MODE_BLOCK) {
        if (wave < 2) {
            rsrc_sf = make_rsrc(sfa_f, (uint32_t)((nk - 1) * p.stride_sfa + p.m) * 4u);
            voff_sf = min(m0 + wave * 64 + lane, p.m - 1) * 4;
            sf_step_bytes = p.stride_sfa * 4;
        } else {
            rsrc_sf = make_rsrc(sfb_f + (long long)(n0 >> 7) * p.stride_sfb, (uint32_t)nk * 4u);
            voff_sf = 0;
            sf_step_bytes = 4;
        }
    }
    // MX: waves 0 and 1 fetch the step's dword (four E8M0 bytes, one per 32 of K) of 64 A rows each, waves 2
    // and 3 those of 64 B rows each
    // (packed E2M1 operands: p.k counts bytes, a row has p.k / 16 scale bytes, eight per K step, fetched as two dwords)
    if constexpr (TALL && (MODE == MODE_MX || MODE == MODE_F4)) {
        // 256-row tiles: every wave fetches those of 64 A rows, and of 64 B rows (waves 2 and 3 the same as 0 and 1)
        const uint32_t row_bytes = MODE == MODE_F4 ? p.k >> 4 : p.k >> 5;
        rsrc_sf = make_rsrc((const uint8_t*)p.sfa + (long long)batch * p.sfa_batch, (uint32_t)(p.m - 1) * p.stride_sfa + row_bytes);
        rsrc_sf_b = make_rsrc((const uint8_t*)p.sfb + (long long)batch * p.sfb_batch, (uint32_t)(p.n - 1) * p.stride_sfb + row_bytes);
        voff_sf = min(m0 + wave * 64 + lane, p.m - 1) * p.stride_sfa;
        voff_sf_b = min(n0 + (wave & 1) * 64 + lane, p.n - 1) * p.stride_sfb;
        sf_step_bytes = MODE == MODE_F4 ? 8 : 4;
    } else if constexpr (MODE == MODE_MX || MODE == MODE_F4) {
        const bool is_b = wave >= 2;
        const int rows = is_b ? p.n : p.m;
        const int stride = is_b ? p.stride_sfb : p.stride_sfa;
        const uint8_t* base = is_b ? (const uint8_t*)p.sfb + (long long)batch * p.sfb_batch
                                   : (const uint8_t*)p.sfa + (long long)batch * p.sfa_batch;
        rsrc_sf = make_rsrc(base, (uint32_t)(rows - 1) * stride + (uint32_t)(MODE == MODE_F4 ? p.k >> 4 : p.k >> 5));
        voff_sf = min((is_b ? n0 : m0) + (wave & 1) * 64 + lane, rows - 1) * stride;
        sf_step_bytes = MODE == MODE_F4 ? 8 : 4;
    }
    // tiled MX: wave w fetches the 512-byte unit of its 64-row block (waves 0, 1: the tile's A blocks, 2, 3: its B
    // blocks) for the step's pair of K steps with one 16-byte load; lanes 32-63 bring the next unit along, unused
    int mxt_nblk = 1, mxt_blk = 0;
    if constexpr (TILED_SCALES) {
        const bool is_b = wave >= 2;
        const int rows = is_b ? p.n : p.m;
        const uint8_t* base = is_b ? (const uint8_t*)p.sfb + (long long)batch * p.sfb_batch
                                   : (const uint8_t*)p.sfa + (long long)batch * p.sfa_batch;
        rsrc_sf = make_rsrc(base, (uint32_t)mx_tiled_bytes(rows, MODE == MODE_F4T ? 2 * p.k : p.k));      // k in elements
        voff_sf = lane * 16;
        mxt_nblk = (rows + 63) >> 6;
        // (a block past the last row: its rows are never stored; a 64-wide tile has one B block, wave 3 brings the next along unused)
        if constexpr (TALL) {
            // 256-row tiles: waves 0 and 1 fetch two units of A each, wave 2 (and 3 once more) the two of B, one per 32 lanes
            const int blk = min(((is_b ? n0 : m0) >> 6) + (is_b ? 0 : 2 * wave) + (lane >> 5), mxt_nblk - 1);
            voff_sf = blk * 1024 + (lane & 31) * 16;
            mxt_blk = 0;
        } else
            mxt_blk = min(((is_b ? n0 : m0) >> 6) + (wave & 1), mxt_nblk - 1);
    }
    // scale load n of a stage
    auto load_scales = [&](int stage, int kstep, int n) __attribute__((always_inline)) {
        if constexpr (TILED_SCALES) {
            A8W8_LDS char* sc = (A8W8_LDS char*)smem + SM_STAGES * SM_STAGE_BYTES + stage * SM_SCALE_BYTES + wave * 1024;
            // the pair of 128-element K steps this step belongs to (FP8: two byte steps) or is (FP4: 256 elements)
            const int pair = MODE == MODE_F4T ? kstep : kstep >> 1;
            load_to_lds_16(rsrc_sf, sc, voff_sf, ((((pair >> 1) * mxt_nblk + mxt_blk) * 2 + (pair & 1)) * 512));
        } else if constexpr (STEP_SCALES) {
            A8W8_LDS char* sc = (A8W8_LDS char*)smem + SM_STAGES * SM_STAGE_BYTES + stage * SM_SCALE_BYTES + wave * 256 + n * 1024;
            // n: 128-row tiles the step's first or second dword (A and B rows), 256-row tiles A's, then B's
            const bool of_b = TALL && n >= SF_LOADS / 2;
            const int dword = (TALL ? n % (SF_LOADS / 2) : n) * 4;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(of_b ? rsrc_sf_b : rsrc_sf, sc, 4, of_b ? voff_sf_b : voff_sf, kstep * sf_step_bytes + dword, 0, 0);
        }
    };
    // Row/col scales of the tile go to LDS behind the stages, in front of the first operand loads (any wait for those covers them), and per-tensor
    // scales to registers, so that the epilogue waits on no load (1600 x 2048 x 1024 8.6 -> 8.3 us,
    // 300 x 3072 x 4096 9.4 -> 9.2, 2560 x 2560 x 1024 12.8 -> 12.6).
    constexpr int ROWCOL_AT = SM_STAGES * (SM_STAGE_BYTES + SM_SCALE_BYTES);
    if constexpr (MODE == MODE_ROWCOL) {
#pragma unroll
        for (int u = 0; u < (SM_BM + SM_BN) / 64; ++u) {
            if (u % 4 != wave) continue;
            const bool of_b = u >= SM_BM / 64;
            const int row = (of_b ? n0 - SM_BM : m0) + 64 * u + lane, rows = of_b ? p.n : p.m;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(of_b ? sfb_f : sfa_f, (uint32_t)rows * 4u), (A8W8_LDS char*)smem + ROWCOL_AT + 256 * u, 4,
                                                     min(row, rows - 1) * 4, 0, 0, 0);
        }
    }
    float ts_a = 1.f, ts_b = 1.f;
    if constexpr (MODE == MODE_TENSOR) {
        ts_a = sfa_f[0];
        ts_b = sfb_f[0];
    }
    auto load_a = [&](A8W8_LDS char* s, int j, int kstep) __attribute__((always_inline)) {
        load_to_lds_16(rsrc_a, s, lane_offset(voff_a[TALL ? 0 : j], kstep), kstep * BK + (TALL ? 32 * j * p.lda : 0));
    };
    auto load_b = [&](A8W8_LDS char* s, int j, int kstep) __attribute__((always_inline)) {
        load_to_lds_16(rsrc_b, s, lane_offset(voff_b[TALL ? 0 : j], kstep), (kstep << p.b_kshift) + (TALL ? 32 * j * p.ldb : 0));
    };
    auto issue_stage = [&](int stage, int kstep) __attribute__((always_inline)) {
        kstep = min(kstep, nk - 1);         // past the end: reload the last step into a stage nobody reads (fixed wait counts)
        A8W8_LDS char* s = (A8W8_LDS char*)smem + stage * SM_STAGE_BYTES + wave * 1024;
#pragma unroll
        for (int j = 0; j < A_LOADS; ++j) load_a(s + j * 4096, j, kstep);
#pragma unroll
        for (int j = 0; j < B_LOADS; ++j) load_b(s + SM_BM * BK + j * 4096, j, kstep);
#pragma unroll
        for (int n = 0; n < SF_LOADS; ++n) load_scales(stage, kstep, n);
    };

    // ---- LDS -> registers: a lane reads K-pieces g and g+4 of tile row r16; slot = piece ^ (row & 7), and
    // row & 7 = lane & 7 for every tile
    int rd_a[2], rd_b[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int slot = (g + 4 * h) ^ (lane & 7);
        rd_a[h] = (wave_m * (SM_BM / 2) + r16) * BK + (slot << 4);
        rd_b[h] = SM_BM * BK + (wave_n * (SM_BN / 2) + r16) * BK + (slot << 4);
    }
    auto read_frag = [&](int stage, const int (&base)[2], int t) __attribute__((always_inline)) -> v8i {
        const char* s = smem + stage * SM_STAGE_BYTES + t * (16 * BK);
        const v4i lo = *(const v4i*)(s + base[0]);
        const v4i hi = *(const v4i*)(s + base[1]);
        return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };

    // tiled MX: byte of (row 16 t + r16 of a 64-row block, 32-block g of the K step, step s of the pair) inside the
    // block's unit, without s (see mx_tiled_index); the same for A tiles and B tiles
    // (a 64-wide tile lies inside one 64-row block of B: wave column 1 owns the block's MFMA tiles 2 and 3)
    int mxt_off[4], mxt_off_b[SM_TN];
    // where the unit of A tile t's 64-row block, and the wave's B block, lie in the stage's scale bytes
    auto mxt_unit_a = [&](int t) __attribute__((always_inline)) { return TALL ? wave_m * 1024 + (t >> 2) * 512 : SHORT ? 0 : wave_m * 1024; };
    const int mxt_unit_b = TALL ? 2048 + wave_n * 512 : SM_BN == 128 ? (2 + wave_n) * 1024 : 2 * 1024;
    constexpr int SF_B_ROW0 = TALL ? (MODE == MODE_F4 ? 512 : 256) : 128;      // dword of B's first row in the row-major scale bytes
    if constexpr (TILED_SCALES) {
        auto unit_offset = [&](int t) __attribute__((always_inline)) {
            const int x = (2 * t + (r16 >> 3)) & 3, y = r16 & 3, par = (r16 >> 2) & 1;
            return ((4 * x + y) * 4 + g) * 8 + (t >> 1) * 4 + par * 2;
        };
#pragma unroll
        for (int t = 0; t < 4; ++t) mxt_off[t] = unit_offset(SHORT ? (2 * wave_m + t) & 3 : t);
#pragma unroll
        for (int t = 0; t < SM_TN; ++t) mxt_off_b[t] = unit_offset(SM_BN == 128 ? t : 2 * wave_n + t);
    }

    const int cm_base = m0 + wave_m * (SM_BM / 2) + r16;          // + 16 * i
    const int cn_base = n0 + wave_n * (SM_BN / 2) + 4 * g;        // + 16 * j + e

    v4f acc[SM_TM][SM_TN];      // (256-row tiles: filled from the accumulation registers behind the K loop)
    if constexpr (!TALL) {
#pragma unroll
        for (int i = 0; i < SM_TM; ++i)
#pragma unroll
            for (int j = 0; j < SM_TN; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    } else {
        asm volatile("" ::: "a0", "a255");      // sizes the wave's register allocation: the compiler has no accumulation registers to itself
    }

    // Deep staging: the step's three instruction streams overlap inside the one wave of a SIMD.  The fragments (and
    // scales) of step ks + 1 are read from LDS while the MFMAs of step ks run (two register sets, the loop unrolled by
    // two), and the stage of step ks -- free as soon as everyone holds its fragments -- is refilled with step
    // ks + SM_STAGES by loads issued one at a time between those MFMAs.  Issued in a block behind the barrier, the loads
    // (which the compute unit's address path takes at 1 KiB per 7 ns), the LDS reads and the MFMAs follow one another:
    // 0.46 us per K step on 128 x 64 tiles where each of the three is 0.11-0.17 us.
    // Two stages (two workgroups per compute unit): there is no third stage to read ahead from, so a step reads all of its
    // fragments first, and behind a second barrier -- the stage is then free -- runs its MFMAs with the refill loads (step
    // ks + 2) between them; the other workgroup's MFMAs run beside this one's LDS reads.
    constexpr bool TWO = SM_STAGES == 2;
    constexpr bool PIPELINED = TWO ? A8W8_SMALL_PIPELINED_TWO != 0 : A8W8_SMALL_PIPELINED != 0;
    static_assert(PIPELINED || (!RAGGED && !TALL && !SHORT), "partial K steps, 256- and 64-row tiles exist in the overlapped loop only");
    if constexpr (PIPELINED) {
        constexpr int HALVES = BY_BF16 ? 4 : (IS_F4 || MODE == MODE_BF16) ? 2 : 1;      // MFMAs per pair of fragments
        constexpr int NFRAG = SM_TM + SM_TN, NSLOT = SM_TM * SM_TN * HALVES, NLOAD = LOADS_PER_STAGE;
        constexpr int LOADS_PER_SLOT = (NLOAD + NSLOT - 1) / NSLOT, LOAD_EVERY = LOADS_PER_SLOT > 1 ? 1 : NSLOT / NLOAD;      // (64 x 64 tiles have fewer MFMAs than loads)
        // converted operands: the next step's first quarter is converted behind this step's last MFMAs, so its fragments come in the first half
        constexpr int READ_EVERY = BY_BF16 && !TWO ? NSLOT / (2 * NFRAG) : NSLOT / NFRAG;
        constexpr int BLK_LAG = MODE == MODE_BLOCK ? 4 : 0;
        static_assert(LOAD_EVERY >= 1 && READ_EVERY >= 1 && (SM_STAGES - 1) * NLOAD < 64, "the wait count is a 6-bit field");
        v8i fr[TWO ? 1 : 2][NFRAG];       // A tiles, then B tiles
        int sc_a[TWO ? 1 : 2][SM_TM], sc_b[TWO ? 1 : 2][SM_TN];      // the step's scales: E8M0 bytes (MX modes), or the A-side factors as float bits (block)
        auto read_one = [&](int stage, int t) __attribute__((always_inline)) -> v8i {
            return t < SM_TM ? read_frag(stage, rd_a, t) : read_frag(stage, rd_b, t - SM_TM);
        };
        auto read_scales = [&](int stage, int ks, int (&sa)[SM_TM], int (&sb)[SM_TN]) __attribute__((always_inline)) {
            const char* sc = smem + SM_STAGES * SM_STAGE_BYTES + stage * SM_SCALE_BYTES;
            if constexpr (MODE == MODE_BLOCK) {
                const float* f = (const float*)sc;
                const float b = f[128];
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) sa[t] = __builtin_bit_cast(int, f[wave_m * (SM_BM / 2) + 16 * t + r16] * b);
            }
            if constexpr (MODE == MODE_MX) {
                // lane (r16, g) scales K [32g, 32g+32) of its row: byte g of the row's dword
                const unsigned* w = (const unsigned*)sc;
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) sa[t] = (int)__builtin_amdgcn_ubfe(w[wave_m * (SM_BM / 2) + 16 * t + r16], 8 * g, 8);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) sb[t] = (int)__builtin_amdgcn_ubfe(w[SF_B_ROW0 + wave_n * (SM_BN / 2) + 16 * t + r16], 8 * g, 8);
            }
            if constexpr (MODE == MODE_F4) {
                // lane (r16, g) scales 32-block g of each 128-element half of its row: byte g of the row's first and of
                // its second dword, put side by side as in the tiled layout (the half is chosen by op_sel)
                const unsigned* w = (const unsigned*)sc;
                auto two_bytes = [&](int row) __attribute__((always_inline)) {
                    return (int)(__builtin_amdgcn_ubfe(w[row], 8 * g, 8) | (__builtin_amdgcn_ubfe(w[256 + row], 8 * g, 8) << 8));
                };
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) sa[t] = two_bytes(wave_m * (SM_BM / 2) + 16 * t + r16);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) sb[t] = two_bytes(SF_B_ROW0 + wave_n * (SM_BN / 2) + 16 * t + r16);
            }
            if constexpr (MODE == MODE_F4T) {
                // both halves' bytes sit side by side: one 16-bit read, the half is chosen by op_sel
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) sa[t] = *(const unsigned short*)(sc + mxt_unit_a(t) + mxt_off[t & 3]);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) sb[t] = *(const unsigned short*)(sc + mxt_unit_b + mxt_off_b[t]);
            }
            if constexpr (MODE == MODE_MXT) {
                const uint8_t* u = (const uint8_t*)sc + (ks & 1);
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) sa[t] = u[mxt_unit_a(t) + mxt_off[t & 3]];
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) sb[t] = u[mxt_unit_b + mxt_off_b[t]];
            }
        };
        // eight E4M3 codes (two dwords: quarter `h` of a fragment) as bf16
        auto quarter_to_bf16 = [&](const v8i& f, int h) __attribute__((always_inline)) -> v8bf {
            const v2bf x0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h], 1.0f, false);
            const v2bf x1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h], 1.0f, true);
            const v2bf x2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h + 1], 1.0f, false);
            const v2bf x3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h + 1], 1.0f, true);
            return v8bf{x0[0], x0[1], x1[0], x1[1], x2[0], x2[1], x3[0], x3[1]};
        };
        // half `part` (two of the four conversions) of the same
        auto half_quarter = [&](v8bf& q, const v8i& f, int h, int part) __attribute__((always_inline)) {
            const v2bf x0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h + part], 1.0f, false);
            const v2bf x1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((unsigned)f[2 * h + part], 1.0f, true);
            q[4 * part] = x0[0]; q[4 * part + 1] = x0[1]; q[4 * part + 2] = x1[0]; q[4 * part + 3] = x1[1];
        };
        v8bf quarter[BY_BF16 ? 2 : 1][NFRAG];      // converted operands: the quarter in use and the next one
        // load n of a stage: the chunks of A, the chunks of B, then the step's scales
        auto load_one = [&](int stage, int kstep, int n) __attribute__((always_inline)) {
            A8W8_LDS char* s = (A8W8_LDS char*)smem + stage * SM_STAGE_BYTES + wave * 1024;
            if (n < A_LOADS) load_a(s + n * 4096, n, kstep);
            else if (n < A_LOADS + B_LOADS) load_b(s + SM_BM * BK + (n - A_LOADS) * 4096, n - A_LOADS, kstep);
            else load_scales(stage, kstep, n - A_LOADS - B_LOADS);
        };
#pragma unroll
        for (int st = 0; st < SM_STAGES; ++st) issue_stage(st, st);
        if constexpr (MODE == MODE_TENSOR) asm volatile("" : "+v"(ts_a), "+v"(ts_b));      // (not fetched where they are used)
        if constexpr (TALL) static_for<SM_TM * SM_TN * 4>([&](auto I) { acc_zero<decltype(I)::value>(); });
        if constexpr (!TWO) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SM_STAGES - 1) * NLOAD) : "memory");
            A8W8_RAW_BARRIER();
#pragma unroll
            for (int t = 0; t < NFRAG; ++t) fr[0][t] = read_one(0, t);
            read_scales(0, 0, sc_a[0], sc_b[0]);
            if constexpr (BY_BF16) {
#pragma unroll
                for (int n = 0; n < NFRAG; ++n) quarter[0][n] = quarter_to_bf16(fr[0][n], 0);
            }
        }
        // one K step: `have`, `sa`, `sb` hold its fragments and scales, the `next_` ones receive those of the step after it
        auto step = [&](int ks, int stage, v8i (&have)[NFRAG], int (&sa)[SM_TM], int (&sb)[SM_TN], v8i (&next)[NFRAG],
                        int (&next_sa)[SM_TM], int (&next_sb)[SM_TN]) __attribute__((always_inline)) {
            const int next_stage = stage + 1 == SM_STAGES ? 0 : stage + 1;
            if constexpr (TWO) {
                // this wave's loads of the step's stage have landed once only the other stage's are in flight; behind the
                // barrier everyone's have
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NLOAD) : "memory");
                A8W8_RAW_BARRIER();
#pragma unroll
                for (int t = 0; t < NFRAG; ++t) have[t] = read_one(stage, t);
                read_scales(stage, ks, sa, sb);
            }
            // this wave's loads of the next step's stage have landed once only the SM_STAGES - 2 younger stages are in
            // flight, and its reads of this step's fragments are complete: behind the barrier both hold for every wave
            if constexpr (!TWO) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SM_STAGES - 2) * NLOAD) : "memory");
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            A8W8_RAW_BARRIER();
            const int kload = min(ks + SM_STAGES, nk - 1);      // past the end: the last step again, into a stage nobody reads
            if constexpr (TALL) {
                // the same order with the accumulators named: a column of eight tiles (two halves of it) at a time
                static_for<NSLOT>([&](auto T) {
                    constexpr int t = decltype(T)::value;
                    constexpr int i = t % SM_TM, h = (t / SM_TM) % HALVES, j = t / (SM_TM * HALVES), lo = 4 * (i * SM_TN + j);
                    const v8i& fb = have[SM_TM + j];
                    const v8i& fa = have[i];
                    if constexpr (IS_F4) {
                        mfma_acc_f4<lo, false, h, h>(v4i{fb[4 * h], fb[4 * h + 1], fb[4 * h + 2], fb[4 * h + 3]},
                                                     v4i{fa[4 * h], fa[4 * h + 1], fa[4 * h + 2], fa[4 * h + 3]}, sb[j], sa[i]);
                    } else if constexpr (MODE == MODE_BF16) {
                        mfma_acc_bf16<lo, false>(v4i{fb[4 * h], fb[4 * h + 1], fb[4 * h + 2], fb[4 * h + 3]},
                                                 v4i{fa[4 * h], fa[4 * h + 1], fa[4 * h + 2], fa[4 * h + 3]});
                    } else if constexpr (MODE == MODE_MX || MODE == MODE_MXT) {
                        mfma_acc_mx<lo, false, 0, 0>(fb, fa, sb[j], sa[i]);
                    } else {
                        mfma_acc<lo, false>(fb, fa);
                    }
                    if constexpr (t % LOAD_EVERY == 0 && t / LOAD_EVERY < NLOAD) load_one(stage, kload, t / LOAD_EVERY);
                    if constexpr (t % READ_EVERY == 0 && t / READ_EVERY < NFRAG) next[t / READ_EVERY] = read_one(next_stage, t / READ_EVERY);
                    if constexpr (t == 0) read_scales(next_stage, ks + 1, next_sa, next_sb);
                    __builtin_amdgcn_sched_barrier(0);
                });
                return next_stage;
            }
            v4f part[BLK_LAG + 1];
            if constexpr (BY_BF16 && TWO) {
#pragma unroll
                for (int n = 0; n < NFRAG; ++n) quarter[0][n] = quarter_to_bf16(have[n], 0);
            }
#pragma unroll
            for (int t = 0; t < NSLOT + BLK_LAG; ++t) {
                if (t < NSLOT) {
                    // fragments pairs column by column; two-MFMA pairs: first halves of the column's four tiles, then second
                    // halves (back-to-back MFMAs on one accumulator stall)
                    // (converted operands: quarter by quarter over all tiles)
                    constexpr int TILES = SM_TM * SM_TN;
                    const int i = t % SM_TM;
                    const int h = BY_BF16 ? t / TILES : (t / SM_TM) % HALVES, j = BY_BF16 ? t % TILES / SM_TM : t / (SM_TM * HALVES);
                    const v8i& fb = have[SM_TM + j];
                    const v8i& fa = have[i];
                    if constexpr (MODE == MODE_BLOCK) {
                        part[t % (BLK_LAG + 1)] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                    } else if constexpr (IS_F4) {
                        // elements [0, 128) of the step sit in the fragments' first 16 bytes, [128, 256) in the second;
                        // op_sel picks the half's scale byte
                        if (h == 0)
                            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                                (v8i{fb[0], fb[1], fb[2], fb[3], 0, 0, 0, 0}), (v8i{fa[0], fa[1], fa[2], fa[3], 0, 0, 0, 0}), acc[i][j], 4, 4, 0,
                                sb[j], 0, sa[i]);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                                (v8i{fb[4], fb[5], fb[6], fb[7], 0, 0, 0, 0}), (v8i{fa[4], fa[5], fa[6], fa[7], 0, 0, 0, 0}), acc[i][j], 4, 4, 1,
                                sb[j], 1, sa[i]);
                    } else if constexpr (MODE == MODE_MX || MODE == MODE_MXT) {
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, acc[i][j], 0, 0, 0, sb[j], 0, sa[i]);
                    } else if constexpr (BY_BF16) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(quarter[h & 1][SM_TM + j], quarter[h & 1][i], acc[i][j], 0, 0, 0);
                        // conversions of the next quarter, spread over this one's MFMAs: one half fragment per MFMA (16 tiles) or two
                        // (8); behind the last quarter those of the next step's first one
                        constexpr int CONV = (2 * NFRAG + TILES - 1) / TILES;
#pragma unroll
                        for (int u = (t % TILES) * CONV; u < (t % TILES + 1) * CONV; ++u) {
                            if (u >= 2 * NFRAG) continue;
                            if (h + 1 < HALVES) half_quarter(quarter[(h + 1) & 1][u >> 1], have[u >> 1], h + 1, u & 1);
                            else if (!TWO) half_quarter(quarter[0][u >> 1], next[u >> 1], 0, u & 1);
                        }
                    } else if constexpr (MODE == MODE_BF16) {
                        // a 128-byte row is 64 bf16: the fragment's two 16-byte halves feed one 16x16x32 MFMA each
                        const v4i bh = {fb[4 * h], fb[4 * h + 1], fb[4 * h + 2], fb[4 * h + 3]};
                        const v4i ah = {fa[4 * h], fa[4 * h + 1], fa[4 * h + 2], fa[4 * h + 3]};
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, bh), __builtin_bit_cast(v8bf, ah), acc[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb, fa, acc[i][j], 0, 0, 0, 0, 0, 0);
                    }
#pragma unroll
                    for (int n = t / LOAD_EVERY * LOADS_PER_SLOT; n < (t / LOAD_EVERY + 1) * LOADS_PER_SLOT; ++n)
                        if (t % LOAD_EVERY == 0 && n < NLOAD) load_one(stage, kload, n);
                    if constexpr (!TWO) {
                        if (t % READ_EVERY == 0 && t / READ_EVERY < NFRAG) next[t / READ_EVERY] = read_one(next_stage, t / READ_EVERY);
                        if (t == 0) read_scales(next_stage, ks + 1, next_sa, next_sb);
                    }
                }
                if constexpr (MODE == MODE_BLOCK) {
                    // acc += part * (sfa * sfb); the multiply-adds trail the MFMAs by BLK_LAG tiles so that they never
                    // wait on a matrix-core result that is still in flight
                    if (t >= BLK_LAG) {
                        const int u = t - BLK_LAG;
                        acc[u % SM_TM][u / SM_TM] += part[u % (BLK_LAG + 1)] * __builtin_bit_cast(float, sa[u % SM_TM]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            return next_stage;
        };
        int ks = 0, stage = 0;
        if constexpr (TWO) {
            for (; ks < nk; ++ks) stage = step(ks, stage, fr[0], sc_a[0], sc_b[0], fr[0], sc_a[0], sc_b[0]);
        } else {
            for (; ks + 1 < nk; ks += 2) {
                stage = step(ks, stage, fr[0], sc_a[0], sc_b[0], fr[1], sc_a[1], sc_b[1]);
                stage = step(ks + 1, stage, fr[1], sc_a[1], sc_b[1], fr[0], sc_a[0], sc_b[0]);
            }
            if (ks < nk) step(ks, stage, fr[0], sc_a[0], sc_b[0], fr[1], sc_a[1], sc_b[1]);
        }
        if constexpr (TALL) {
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // last MFMA -> first accumulator read
            static_for<SM_TM * SM_TN>([&](auto IJ) {
                constexpr int ij = decltype(IJ)::value;
                static_for<4>([&](auto E) { acc[ij / SM_TN][ij % SM_TN][decltype(E)::value] = acc_read<4 * ij + decltype(E)::value>(); });
            });
        }
    } else {
    issue_stage(0, 0);
    issue_stage(1, 1);
    if constexpr (SM_STAGES > 2) {
#pragma unroll
        for (int st = 2; st < SM_STAGES - 1; ++st) issue_stage(st, st);
    }
    // stages in flight behind the one being read: one of two, else all but the one being refilled
    constexpr int YOUNGER = SM_STAGES == 2 ? 1 : SM_STAGES - 2;
    static_assert(YOUNGER * LOADS_PER_STAGE < 64, "the wait count is a 6-bit field");

    int cur = 0, refill = SM_STAGES - 1;      // the stage of step ks, the stage of step ks - 1 (refilled with step ks + SM_STAGES - 1)
    for (int ks = 0; ks < nk; ++ks) {
        // this wave's loads of stage `cur` have landed once only the younger stages are in flight
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER * LOADS_PER_STAGE) : "memory");
        A8W8_RAW_BARRIER();                 // ... everyone's have; and (more than two stages) everyone is done reading the stage of step ks-1
        if constexpr (SM_STAGES > 2) issue_stage(refill, ks + SM_STAGES - 1);

        v8i fa[SM_TM], fb[2];
#pragma unroll
        for (int t = 0; t < SM_TM; ++t) fa[t] = read_frag(cur, rd_a, t);
        fb[0] = read_frag(cur, rd_b, 0);
        if constexpr (MODE == MODE_BLOCK) {
            const float* sc = (const float*)(smem + SM_STAGES * SM_STAGE_BYTES + cur * SM_SCALE_BYTES);
            const float sb = sc[128];
            float blk_s[SM_TM];
#pragma unroll
            for (int t = 0; t < SM_TM; ++t) blk_s[t] = sc[wave_m * 64 + 16 * t + r16] * sb;
            // acc += part * (sfa * sfb); the multiply-adds trail the MFMAs by BLK_LAG tiles so that they never
            // wait on a matrix-core result that is still in flight
            constexpr int BLK_LAG = 4;
            v4f part[BLK_LAG + 1];
#pragma unroll
            for (int t = 0; t < SM_TM * SM_TN + BLK_LAG; ++t) {
                if (t < SM_TM * SM_TN) {
                    const int j = t / SM_TM, i = t % SM_TM;
                    if (i == 0 && j + 1 < SM_TN) fb[(j + 1) & 1] = read_frag(cur, rd_b, j + 1);
                    part[t % (BLK_LAG + 1)] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        fb[j & 1], fa[i], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);   // keep the lag: the scheduler would pull the FMAs up
                if (t >= BLK_LAG) {
                    const int u = t - BLK_LAG;
                    acc[u % SM_TM][u / SM_TM] += part[u % (BLK_LAG + 1)] * blk_s[u % SM_TM];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            int mx_sa[SM_TM], mx_sb[SM_TN];
            if constexpr (MODE == MODE_MX) {
                // lane (r16, g) scales K [32g, 32g+32) of its row: byte g of the row's dword
                const unsigned* sc = (const unsigned*)(smem + SM_STAGES * SM_STAGE_BYTES + cur * SM_SCALE_BYTES);
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) mx_sa[t] = (int)__builtin_amdgcn_ubfe(sc[wave_m * 64 + 16 * t + r16], 8 * g, 8);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) mx_sb[t] = (int)__builtin_amdgcn_ubfe(sc[128 + wave_n * (SM_BN / 2) + 16 * t + r16], 8 * g, 8);
            }
            if constexpr (MODE == MODE_F4) {
                // lane (r16, g) scales 32-block g of each 128-element half of its row: byte g of the row's first and of
                // its second dword, put side by side as in the tiled layout (the half is chosen by op_sel)
                const unsigned* sc = (const unsigned*)(smem + SM_STAGES * SM_STAGE_BYTES + cur * SM_SCALE_BYTES);
                auto two_bytes = [&](int row) __attribute__((always_inline)) {
                    return (int)(__builtin_amdgcn_ubfe(sc[row], 8 * g, 8) | (__builtin_amdgcn_ubfe(sc[256 + row], 8 * g, 8) << 8));
                };
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) mx_sa[t] = two_bytes(wave_m * (SM_BM / 2) + 16 * t + r16);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) mx_sb[t] = two_bytes(SF_B_ROW0 + wave_n * (SM_BN / 2) + 16 * t + r16);
            }
            if constexpr (MODE == MODE_F4T) {
                // both halves' bytes sit side by side: one 16-bit read, the half is chosen by op_sel
                const char* sc = smem + SM_STAGES * SM_STAGE_BYTES + cur * SM_SCALE_BYTES;
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) mx_sa[t] = *(const unsigned short*)(sc + wave_m * 1024 + mxt_off[t]);
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) mx_sb[t] = *(const unsigned short*)(sc + mxt_unit_b + mxt_off_b[t]);
            }
            if constexpr (MODE == MODE_MXT) {
                const uint8_t* sc = (const uint8_t*)(smem + SM_STAGES * SM_STAGE_BYTES + cur * SM_SCALE_BYTES) + (ks & 1);
#pragma unroll
                for (int t = 0; t < SM_TM; ++t) mx_sa[t] = sc[wave_m * 1024 + mxt_off[t]];
#pragma unroll
                for (int t = 0; t < SM_TN; ++t) mx_sb[t] = sc[mxt_unit_b + mxt_off_b[t]];
            }
#pragma unroll
            for (int j = 0; j < SM_TN; ++j) {
                if (j + 1 < SM_TN) fb[(j + 1) & 1] = read_frag(cur, rd_b, j + 1);
                if constexpr (IS_F4) {
                    // two FP4 MFMAs per fragment pair: elements [0, 128) of the step sit in the fragments' first 16
                    // bytes, [128, 256) in the second; op_sel picks the half's scale byte
#pragma unroll
                    for (int i = 0; i < SM_TM; ++i) {
                        const v8i& fbj = fb[j & 1];
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                            (v8i{fbj[0], fbj[1], fbj[2], fbj[3], 0, 0, 0, 0}), (v8i{fa[i][0], fa[i][1], fa[i][2], fa[i][3], 0, 0, 0, 0}),
                            acc[i][j], 4, 4, 0, mx_sb[j], 0, mx_sa[i]);
                    }
#pragma unroll
                    for (int i = 0; i < SM_TM; ++i) {
                        const v8i& fbj = fb[j & 1];
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                            (v8i{fbj[4], fbj[5], fbj[6], fbj[7], 0, 0, 0, 0}), (v8i{fa[i][4], fa[i][5], fa[i][6], fa[i][7], 0, 0, 0, 0}),
                            acc[i][j], 4, 4, 1, mx_sb[j], 1, mx_sa[i]);
                    }
                } else if constexpr (MODE == MODE_MX || MODE == MODE_MXT) {
#pragma unroll
                    for (int i = 0; i < SM_TM; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j & 1], fa[i], acc[i][j], 0, 0, 0, mx_sb[j], 0,
                                                                                     mx_sa[i]);
                } else if constexpr (MODE == MODE_BF16) {
                    // a 128-byte row is 64 bf16: the fragment's two 16-byte halves feed one 16x16x32 MFMA each (both
                    // operands split K the same way); first halves for all four tiles, then second halves:
                    // back-to-back MFMAs on one accumulator stall
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int i = 0; i < SM_TM; ++i) {
                            const v8i& fbj = fb[j & 1];
                            const v4i bh = {fbj[4 * h], fbj[4 * h + 1], fbj[4 * h + 2], fbj[4 * h + 3]};
                            const v4i ah = {fa[i][4 * h], fa[i][4 * h + 1], fa[i][4 * h + 2], fa[i][4 * h + 3]};
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, bh), __builtin_bit_cast(v8bf, ah),
                                                                                acc[i][j], 0, 0, 0);
                        }
                } else {
#pragma unroll
                    for (int i = 0; i < SM_TM; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j & 1], fa[i], acc[i][j], 0, 0, 0, 0, 0, 0);
                }
            }
        }
        if constexpr (SM_STAGES == 2) {
            // everyone is done reading stage `cur`: refill it with the step after next (the next step's wait lets
            // exactly these loads stay in flight)
            A8W8_RAW_BARRIER();
            issue_stage(cur, ks + 2);
        }
        refill = cur;
        cur = cur + 1 == SM_STAGES ? 0 : cur + 1;
    }
    }

    // ---- epilogue: dequantise in fp32, convert, store
    float sa[SM_TM];
    const float ts = ts_a * ts_b;
    const float* row_scales = (const float*)(smem + ROWCOL_AT);      // the tile's rows, then its columns
    if constexpr (MODE == MODE_ROWCOL) {
#pragma unroll
        for (int i = 0; i < SM_TM; ++i) sa[i] = row_scales[cm_base - m0 + 16 * i];
    }
    char* c_base = (char*)p.c + (long long)batch * p.c_batch * (CDT == C_BF16 ? 2 : 4);
    const bool vec_ok = (CDT == C_BF16) ? ((p.ldc & 3) == 0 && (((uintptr_t)c_base) & 7) == 0)
                                        : ((p.ldc & 3) == 0 && (((uintptr_t)c_base) & 15) == 0);
    const bool whole = vec_ok && m0 + SM_BM <= p.m && n0 + SM_BN <= p.n;
#if A8W8_SMALL_LINES_BY_LANE
    // A tile leaves through LDS, 16 rows of the wave's 64 at a time: the MFMA layout's stores have
    // neighbouring lanes in different rows (16 rows x 16 bytes per 16 lanes), which occupies the memory pipeline 2.7 times as long as
    // stores whose consecutive lanes write consecutive 16 bytes of a row.  A problem of few tiles ends with every workgroup's stores
    // and nothing to hide them behind.  The wave writes the 16 x (16 SM_TN) values into its own 4.25 KiB of LDS (rows padded
    // by 16 bytes against bank conflicts), reads them back along the rows and stores 16 bytes per lane; a wave's LDS
    // operations complete in order, so neither step needs a barrier.  Every direct-to-LDS load has landed by then (the
    // loop's last loads re-fill stages nobody reads).
    // Tiles on the edge of the matrix too, as long as the matrix ends on one of the 16-byte pieces: a lane stores its piece or
    // not.  (From the MFMA layout, with checks per element, they ended after all others: row/col 1000 x 3000, K = 512: 8.2 us against 6.3
    // on 1024 x 3072, 6.7 this way; K = 2048 12.4 -> 10.9, 10.4 on 1024 x 3072.)
    constexpr int ES = CDT == C_BF16 ? 2 : 4;
    auto write_lines = [&](auto CHECKED) __attribute__((always_inline)) {
        constexpr bool checked = decltype(CHECKED)::value != 0;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        constexpr int ROW_BYTES = SM_TN * 16 * ES;                 // the wave's columns of one row
        constexpr int ROW_PITCH = ROW_BYTES + 16;
        constexpr int LANES_PER_ROW = ROW_BYTES / 16, ROWS_PER_STORE = 64 / LANES_PER_ROW, STORES = 16 / ROWS_PER_STORE;
        char* mine = smem + wave * (16 * (SM_BN / 2 * 4 + 16));
        const int wr = r16 * ROW_PITCH + 4 * g * ES;              // + 16 j ES: the lane's four values of MFMA tile j
        const int rd = (lane / LANES_PER_ROW) * ROW_PITCH + (lane % LANES_PER_ROW) * 16;      // + ROWS_PER_STORE rows per store
        char* c_wave = c_base + ((long long)(m0 + wave_m * (SM_BM / 2)) * p.ldc + n0 + wave_n * (SM_BN / 2)) * ES;
        const long long row_bytes = (long long)p.ldc * ES;
        // rows of the wave's part that exist below the lane's first one (none where its piece's columns do not)
        const int rows_left = n0 + wave_n * (SM_BN / 2) + (lane % LANES_PER_ROW) * (16 / ES) < p.n
                                  ? p.m - (m0 + wave_m * (SM_BM / 2)) - lane / LANES_PER_ROW : 0;
        v4f sb_all[SM_TN];
        if constexpr (MODE == MODE_ROWCOL) {
#pragma unroll
            for (int j = 0; j < SM_TN; ++j) sb_all[j] = *(const v4f*)(row_scales + SM_BM + (cn_base - n0) + 16 * j);
        }
#pragma unroll
        for (int i = 0; i < SM_TM; ++i) {
#pragma unroll
            for (int j = 0; j < SM_TN; ++j) {
                v4f v = acc[i][j];
                if constexpr (MODE == MODE_TENSOR) v *= ts;
                if constexpr (MODE == MODE_ROWCOL) v *= sb_all[j] * sa[i];
                if constexpr (CDT == C_BF16) *(v2i*)(mine + wr + 16 * j * ES) = v2i{bf16x2_bits(v.x, v.y), bf16x2_bits(v.z, v.w)};
                else *(v4f*)(mine + wr + 16 * j * ES) = v;
            }
#pragma unroll
            for (int st = 0; st < STORES; ++st) {
                const v4i w = *(const v4i*)(mine + rd + st * ROWS_PER_STORE * ROW_PITCH);
                const int row = 16 * i + st * ROWS_PER_STORE + lane / LANES_PER_ROW;
                if (!checked || 16 * i + st * ROWS_PER_STORE < rows_left) A8W8_STORE_C((v4i*)(c_wave + row * row_bytes + (lane % LANES_PER_ROW) * 16), w);
            }
        }
    };
    if ((n0 + SM_BN <= p.n || (p.n & (16 / ES - 1)) == 0) && (p.ldc & (16 / ES - 1)) == 0 && (((uintptr_t)c_base) & 15) == 0) {
        if (whole) write_lines(std::integral_constant<int, 0>{});
        else write_lines(std::integral_constant<int, 1>{});
        return;
    }
#endif
#pragma unroll
    for (int j = 0; j < SM_TN; ++j) {
        const int cn = cn_base + 16 * j;
        v4f sb = v4f{1.f, 1.f, 1.f, 1.f};
        if constexpr (MODE == MODE_ROWCOL) sb = *(const v4f*)(row_scales + SM_BM + (cn - n0));
#pragma unroll
        for (int i = 0; i < SM_TM; ++i) {
            const int cm = cm_base + 16 * i;
            v4f v = acc[i][j];
            if constexpr (MODE == MODE_TENSOR) v *= ts;
            if constexpr (MODE == MODE_ROWCOL) v *= sb * sa[i];
            if (whole) {        // inside the matrix, aligned rows: no per-lane checks
                if constexpr (CDT == C_BF16)
                    A8W8_STORE_C((v2i*)((unsigned short*)c_base + (long long)cm * p.ldc + cn), (v2i{bf16x2_bits(v.x, v.y), bf16x2_bits(v.z, v.w)}));
                else
                    A8W8_STORE_C((v4f*)((float*)c_base + (long long)cm * p.ldc + cn), v);
                continue;
            }
            if (cm >= p.m) continue;
            if constexpr (CDT == C_BF16) {
                unsigned short* dst = (unsigned short*)c_base + (long long)cm * p.ldc + cn;
                if (vec_ok && cn + 3 < p.n) {
                    A8W8_STORE_C((v2i*)dst, (v2i{bf16x2_bits(v.x, v.y), bf16x2_bits(v.z, v.w)}));
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (cn + e < p.n) dst[e] = bf16_bits(v[e]);
                }
            } else {
                float* dst = (float*)c_base + (long long)cm * p.ldc + cn;
                if (vec_ok && cn + 3 < p.n) {
                    A8W8_STORE_C((v4f*)dst, v);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (cn + e < p.n) dst[e] = v[e];
                }
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct-to-LDS load may outlive the workgroup's LDS allocation
}

}  // namespace a8w8
