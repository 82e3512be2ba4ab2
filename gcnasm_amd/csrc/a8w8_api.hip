// C ABI of libmi355a8w8: argument validation, kernel selection, launches.
#include "../../include/mi355_a8w8.h"

#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <mutex>
#include <tuple>
#include <utility>

#include "cvt.hpp"
#include "flatmm.hpp"
#include "gemm_general.hpp"
#include "gemm_persist.hpp"
#include "gemm_small.hpp"
#include "gemm_wide.hpp"
#include "hbm_probe.hpp"
#include "routes.hpp"

using namespace a8w8;

namespace {

// ---------------------------------------------------------------- per-device set-up, done once
// What a device needs before its first launch: its architecture and compute-unit count, and the
// dynamic-LDS limit of every kernel instantiation that uses more than the 64 KiB default.  It runs
// exactly once per device (std::call_once: concurrent first calls from several threads wait for
// it), either from a8w8_init or from the first entry point called with that device current.
constexpr int MAX_DEVICES = 64;
struct DeviceState {
    std::once_flag once;
    int status = A8W8_ERR_NO_DEVICE;
    int num_cus = 0;
};
DeviceState g_dev[MAX_DEVICES];

template <class K>
bool raise_lds_limit(K kern, int bytes)
{
    return hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
}

constexpr int persist_lds_bytes(int mode)
{
    return mode == MODE_MX ? PERSIST_LDS_BYTES_MX : mode == MODE_ROWCOL ? PERSIST_LDS_BYTES_ROWCOL : PERSIST_LDS_BYTES;
}

// LDS stages of the 128 x 64 variant of the 128-tile kernel: three, and as many as fit 160 KiB (narrow_tiles_deep)
constexpr int NARROW_STAGES = 3, SHORT_STAGES = 4;      // (64 x 64 tiles: four; six and eight are 2 to 10% slower)
constexpr int narrow_deep_stages(int mode) { return mode == MODE_MXT || mode == MODE_F4T ? 5 : 6; }

template <int MODE>
bool raise_lds_limits_of_mode()
{
    bool ok = true;
    if constexpr (MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_BLOCK || MODE == MODE_MX || MODE == MODE_BF16)
        ok = ok && raise_lds_limit(gemm_a8w8_persist<MODE, C_BF16>, persist_lds_bytes(MODE)) &&
             raise_lds_limit(gemm_a8w8_persist<MODE, C_FP32>, persist_lds_bytes(MODE));
    if constexpr (MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_MXT || MODE == MODE_MX || MODE == MODE_BF16 || MODE == MODE_F4T || MODE == MODE_F4)
        ok = ok && raise_lds_limit(gemm_a8w8_wide<MODE, C_BF16>, wide_lds_bytes(MODE)) &&
             raise_lds_limit(gemm_a8w8_wide<MODE, C_FP32>, wide_lds_bytes(MODE));
    {
        ok = ok && raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, 2>, small_lds_bytes(MODE, 2)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, 2>, small_lds_bytes(MODE, 2)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, 4>, small_lds_bytes(MODE, 4)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, 4>, small_lds_bytes(MODE, 4)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, NARROW_STAGES, 64>, small_lds_bytes(MODE, NARROW_STAGES, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, NARROW_STAGES, 64>, small_lds_bytes(MODE, NARROW_STAGES, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, SHORT_STAGES, 64, false, 64>, small_lds_bytes(MODE, SHORT_STAGES, 64, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, SHORT_STAGES, 64, false, 64>, small_lds_bytes(MODE, SHORT_STAGES, 64, 64));
    }
    constexpr int deep = narrow_deep_stages(MODE);
    ok = ok && raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, deep, 64>, small_lds_bytes(MODE, deep, 64)) &&
         raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, deep, 64>, small_lds_bytes(MODE, deep, 64));
    if constexpr (MODE != MODE_BLOCK)
        ok = ok && raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, 3, SM_BN, false, 256>, small_lds_bytes(MODE, 3, SM_BN, 256)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, 3, SM_BN, false, 256>, small_lds_bytes(MODE, 3, SM_BN, 256));
    if constexpr (MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_BF16)
        ok = ok && raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, 2, SM_BN, true>, small_lds_bytes(MODE, 2)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, 2, SM_BN, true>, small_lds_bytes(MODE, 2)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, 4, SM_BN, true>, small_lds_bytes(MODE, 4)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, 4, SM_BN, true>, small_lds_bytes(MODE, 4)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, NARROW_STAGES, 64, true>, small_lds_bytes(MODE, NARROW_STAGES, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, NARROW_STAGES, 64, true>, small_lds_bytes(MODE, NARROW_STAGES, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, deep, 64, true>, small_lds_bytes(MODE, deep, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, deep, 64, true>, small_lds_bytes(MODE, deep, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_BF16, SHORT_STAGES, 64, true, 64>, small_lds_bytes(MODE, SHORT_STAGES, 64, 64)) &&
             raise_lds_limit(gemm_a8w8_tile128<MODE, C_FP32, SHORT_STAGES, 64, true, 64>, small_lds_bytes(MODE, SHORT_STAGES, 64, 64));
    return ok;
}

// runs with device `dev` current
void set_up_device(int dev)
{
    DeviceState& d = g_dev[dev];
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) { d.status = A8W8_ERR_NO_DEVICE; return; }
    d.num_cus = prop.multiProcessorCount;
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) { d.status = A8W8_ERR_NO_DEVICE; return; }
    const bool ok = raise_lds_limits_of_mode<MODE_TENSOR>() && raise_lds_limits_of_mode<MODE_ROWCOL>() &&
                    raise_lds_limits_of_mode<MODE_BLOCK>() && raise_lds_limits_of_mode<MODE_MX>() &&
                    raise_lds_limits_of_mode<MODE_MXT>() && raise_lds_limits_of_mode<MODE_BF16>() &&
                    raise_lds_limits_of_mode<MODE_F4T>() && raise_lds_limits_of_mode<MODE_F4>();
    d.status = ok ? A8W8_OK : A8W8_ERR_LAUNCH;
}

// A8W8_OK when the current device is a gfx950 that has been set up (setting it up on first use).
int device_status()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return A8W8_ERR_NO_DEVICE;
    std::call_once(g_dev[dev].once, set_up_device, dev);
    return g_dev[dev].status;
}

// One kernel launch; the status is that of this launch alone (hipLaunchKernel's own return value, not the
// thread's sticky last error, which an earlier unrelated runtime call may have set).
template <class... P, class... A, size_t... I>
int launch_impl(void (*kern)(P...), dim3 grid, dim3 block, unsigned lds, hipStream_t s, std::index_sequence<I...>, A&&... a)
{
    std::tuple<P...> params{static_cast<P>(std::forward<A>(a))...};
    void* ptrs[] = {(void*)&std::get<I>(params)...};
    return hipLaunchKernel((const void*)kern, grid, block, ptrs, lds, s) == hipSuccess ? A8W8_OK : A8W8_ERR_LAUNCH;
}
template <class... P, class... A>
int launch(void (*kern)(P...), dim3 grid, dim3 block, unsigned lds, hipStream_t s, A&&... a)
{
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    return launch_impl(kern, grid, block, lds, s, std::index_sequence_for<P...>{}, std::forward<A>(a)...);
}
// a launch in the middle of a sequence: leave with its status if it failed
#define A8W8_LAUNCH_OR_RETURN(...)                       \
    do {                                                 \
        const int st_ = launch(__VA_ARGS__);             \
        if (st_ != A8W8_OK) return st_;                  \
    } while (0)

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The two pipelined kernels (and only they) address the 256 rows of a C tile with unsigned 32-bit byte offsets from
// the tile's origin: (255 stride_c + 256) elements of `elem_bytes` must stay below 2^32.  That is stride_c up to
// 4,210,751 for fp32 and 8,421,503 for bf16; the other kernels address C with 64-bit pointers and take any stride.
bool c_tile_fits(long long stride_c, int elem_bytes)
{
    return ((long long)(BM - 1) * stride_c + BN) * elem_bytes < (1ll << 32);
}

// Checks shared by every GEMM entry point (mirrors the reference harness's rejects,
// gemm_a8w8_blockscale_host.cc:175-187, and adds the pointer/stride checks a library needs).
int validate_common(const a8w8_gemm_args* g)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    if (!g->a || !g->b || !g->c || !g->sfa || !g->sfb) return A8W8_ERR_NULL_POINTER;
    if (g->m <= 0 || g->n <= 0 || g->k <= 0 || g->batch <= 0) return A8W8_ERR_BAD_SHAPE;
    if (g->scale_mode < 0 || g->scale_mode > A8W8_SCALE_MX_E8M0_TILED) return A8W8_ERR_BAD_MODE;
    if (g->c_dtype != A8W8_C_BF16 && g->c_dtype != A8W8_C_FP32) return A8W8_ERR_BAD_MODE;
    if (g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128 && (g->n % 128 != 0 || g->k % 128 != 0))
        return A8W8_ERR_BAD_GROUP;
    if ((g->scale_mode == A8W8_SCALE_MX_E8M0_1x32 || g->scale_mode == A8W8_SCALE_MX_E8M0_TILED) && g->k % 32 != 0)
        return A8W8_ERR_BAD_GROUP;
    if (g->stride_c < g->n) return A8W8_ERR_BAD_STRIDE;
    if (g->stride_a < g->k) return A8W8_ERR_BAD_STRIDE;
    if (!g->b_preshuffled && g->stride_b < g->k) return A8W8_ERR_BAD_STRIDE;
    if (g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128 && (g->stride_sfa < g->m || g->stride_sfb < g->k / 128))
        return A8W8_ERR_BAD_STRIDE;
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_1x32 && (g->stride_sfa < g->k / 32 || g->stride_sfb < g->k / 32))
        return A8W8_ERR_BAD_STRIDE;
    if (g->batch > 1 && (g->stride_a_batch < 0 || g->stride_b_batch < 0 || g->stride_c_batch < 0 ||
                         g->stride_sfa_batch < 0 || g->stride_sfb_batch < 0))
        return A8W8_ERR_BAD_STRIDE;
    // the kernels address one batch of A / B with 32-bit byte offsets
    const long long a_span = (long long)(g->m - 1) * g->stride_a + g->k;
    const long long b_span = g->b_preshuffled ? (long long)g->n * g->k : (long long)(g->n - 1) * g->stride_b + g->k;
    if (a_span >= (1ll << 31) || b_span >= (1ll << 31)) return A8W8_ERR_TOO_LARGE;
    if (g->batch > 65535) return A8W8_ERR_TOO_LARGE;
    // ... and the A-side block scales of all K groups, and count 128 x 128 tiles with an int
    if (g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128 && (long long)(g->k / 128) * g->stride_sfa * 4 >= (1ll << 31))
        return A8W8_ERR_TOO_LARGE;
    if ((long long)((g->m + 127) / 128) * ((g->n + 127) / 128) >= (1ll << 31)) return A8W8_ERR_TOO_LARGE;
    return A8W8_OK;
}

GemmParams make_params(const a8w8_gemm_args* g)
{
    GemmParams p;
    p.a = (const uint8_t*)g->a;
    p.b = (const uint8_t*)g->b;
    p.c = g->c;
    p.sfa = g->sfa;
    p.sfb = g->sfb;
    p.m = g->m; p.n = g->n; p.k = g->k;
    p.lda = g->stride_a; p.ldc = g->stride_c;
    // pre-shuffled B: 16 rows span 16 k bytes and a 128-wide K step two 1 KiB blocks
    p.ldb = g->b_preshuffled ? g->k : g->stride_b;
    p.b_kshift = g->b_preshuffled ? 11 : 7;
    p.a_batch = g->stride_a_batch; p.b_batch = g->stride_b_batch; p.c_batch = g->stride_c_batch;
    p.sfa_batch = g->stride_sfa_batch; p.sfb_batch = g->stride_sfb_batch;
    p.stride_sfa = g->stride_sfa; p.stride_sfb = g->stride_sfb;
    p.tiles_m = (g->m + BM - 1) / BM;
    p.tiles_n = (g->n + BN - 1) / BN;
    p.inv_per_group = p.inv_rem = 0;
    p.runs = 0;
    return p;
}

// 16-byte aligned rows in A and B.
bool rows_aligned(const a8w8_gemm_args* g)
{
    return g->stride_a % 16 == 0 && g->stride_b % 16 == 0 && aligned16(g->a) && aligned16(g->b) &&
           (g->batch == 1 || (g->stride_a_batch % 16 == 0 && g->stride_b_batch % 16 == 0));
}

// The tiled kernels need whole 128-wide K steps and 16-byte aligned rows in A and B; the MX
// variant also stages its scale bytes with dword-granular loads.
bool tiled_ok(const a8w8_gemm_args* g)
{
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_1x32 &&
        (g->stride_sfa % 4 != 0 || g->stride_sfb % 4 != 0 || ((uintptr_t)g->sfa & 3) || ((uintptr_t)g->sfb & 3) ||
         (g->batch > 1 && (g->stride_sfa_batch % 4 != 0 || g->stride_sfb_batch % 4 != 0))))
        return false;
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_TILED &&
        (!aligned16(g->sfa) || !aligned16(g->sfb) ||
         (g->batch > 1 && (g->stride_sfa_batch % 16 != 0 || g->stride_sfb_batch % 16 != 0))))
        return false;
    return g->k % BK == 0 && rows_aligned(g) && (long long)((g->m + BM - 1) / BM) * ((g->n + BN - 1) / BN) < (1ll << 31);
}

// The 128-tile kernel with a partial last K step: rows of whole 16-byte pieces, scales that do not change with K (k in bytes here).
bool ragged_ok(const a8w8_gemm_args* g)
{
    return (g->scale_mode == A8W8_SCALE_TENSOR || g->scale_mode == A8W8_SCALE_ROWCOL) && !g->b_preshuffled && g->k % BK != 0 &&
           g->k % 16 == 0 && rows_aligned(g) && (long long)((g->m + SM_BM - 1) / SM_BM) * ((g->n + 63) / 64) < (1ll << 31) &&
           partial_steps_on_tiles(g->m, g->n, g->k, g->batch);
}

// B in the a8w8_preshuffle_b layout is read by the MFMA kernels only (the one-thread-per-element kernel reads
// row-major B): whole 16-row groups and 128-wide K steps, aligned pointers.
int validate_shuffled_b(const a8w8_gemm_args* g)
{
    if (!g->b_preshuffled) return A8W8_OK;
    if (g->n % 16 != 0 || g->k % BK != 0) return A8W8_ERR_BAD_GROUP;
    a8w8_gemm_args rows = *g;
    rows.stride_b = g->k;           // what the alignment checks of tiled_ok should see for B
    return tiled_ok(&rows) ? A8W8_OK : A8W8_ERR_MISALIGNED;
}

int num_cus();

// What the pipelined kernels count with an int: two K steps at least, the work items.
bool items_ok(const a8w8_gemm_args* g)
{
    return g->k >= 2 * BK && (long long)g->batch * ((g->m + BM - 1) / BM) * ((g->n + BN - 1) / BN) < (1ll << 30);
}

// Whether the four-wave kernel takes the number of K steps: any even one, odd ones where odd_steps_on_four_waves and
// odd_tiled_mx_on_four_waves say so.  (Tiled scales with an odd number and C rows too far apart for its 32-bit offsets stay with the 128-tile
// kernel, which takes any distance.)  `fp4`: the byte view of packed E2M1 operands.
bool steps_on_four_waves(const a8w8_gemm_args* g, bool fp4)
{
    const int steps = g->k / BK;
    if (steps % 2 == 0) return true;
    if (g->scale_mode != A8W8_SCALE_MX_E8M0_TILED) return odd_steps_on_four_waves(steps);
    const bool fp32 = g->c_dtype == A8W8_C_FP32;
    return odd_tiled_mx_on_four_waves(fp4, g->m, g->n, steps, g->batch, fp32, num_cus()) && c_tile_fits(g->stride_c, fp32 ? 4 : 2) && items_ok(g);
}

// The persistent kernels; tiled MX scales exist on the four-wave one only.
bool persist_ok(const a8w8_gemm_args* g, bool fp4 = false)
{
    return items_ok(g) && (g->scale_mode != A8W8_SCALE_MX_E8M0_TILED || steps_on_four_waves(g, fp4));
}

// The four-wave kernel has every scale mode but block scales.  Row-major MX scales: 32-bit offsets that run up to 256 rows past the end of the
// matrix.
bool wide_ok(const a8w8_gemm_args* g)
{
    if (g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128) return false;
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_1x32)
        return items_ok(g) && mx_row_scales_on_four_waves(g->k / BK) && (g->m + (long long)BM) * g->stride_sfa < (1ll << 31) &&
               (g->n + (long long)BM) * g->stride_sfb < (1ll << 31);
    return items_ok(g) && steps_on_four_waves(g, false);
}

bool small_ok(const a8w8_gemm_args* g, bool fp4 = false);

// MXFP4 with row-major scales on the four-wave kernel (`g`: byte view, k in bytes, row-major scale mode).  It fetches 16 scale
// bytes of a row at a time (two K steps) with 32-bit offsets that run up to 256 rows past the end of the matrix.  Scale rows of an odd number of
// steps are eight bytes more than a multiple of 16, and its loads then start on dwords, as the caller has checked.  Up to two 128-tiles per
// compute unit (fits_128_tiles, the line of every other mode) and where f4_row_scales_on_256_tiles says so the 128-tile kernel is the faster one.
bool wide_row_scales_ok(const a8w8_gemm_args* g)
{
    const bool odd = (g->k / BK) % 2 != 0;
    const auto rows_ok = [&](const void* s, long long stride, long long batch_stride, long long rows) {
        return (odd || (aligned16(s) && stride % 16 == 0 && (g->batch == 1 || batch_stride % 16 == 0))) && (rows + BM) * stride < (1ll << 31);
    };
    return !fits_128_tiles(g->m, g->n, g->batch, num_cus()) && f4_row_scales_on_256_tiles(g->m, g->n, g->k / BK, g->batch, g->c_dtype == A8W8_C_FP32, num_cus()) &&
           items_ok(g) && rows_ok(g->sfa, g->stride_sfa, g->stride_sfa_batch, g->m) &&
           rows_ok(g->sfb, g->stride_sfb, g->stride_sfb_batch, g->n) && c_tile_fits(g->stride_c, g->c_dtype == A8W8_C_BF16 ? 2 : 4);
}

template <int MODE, int CDT>
int launch_general(const GemmParams& p, int batch, hipStream_t stream);

// compute units of the current device (256 before the device has been set up: kernel-name queries on a CPU box)
int num_cus()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return 256;
    return g_dev[dev].num_cus > 0 ? g_dev[dev].num_cus : 256;
}

// Two 128-tiles per compute unit at most (fits_128_tiles), or rounds of 256-tiles that leave the chip idle (rounds_on_128_tiles).
bool small_ok(const a8w8_gemm_args* g, bool fp4)
{
    const bool mxt = g->scale_mode == A8W8_SCALE_MX_E8M0_TILED;
    // tiled MX scales on a number of K steps that the four-wave kernel does not take have no other kernel: any size runs here
    if (mxt && !steps_on_four_waves(g, fp4)) return true;
    // (C rows too far apart for the 256-tile kernels stay refused)
    const bool fp32 = g->c_dtype == A8W8_C_FP32;
    const RoundsKind kind = mxt ? (fp4 ? ROUNDS_MXFP4_TILED : ROUNDS_MXFP8_TILED) : g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128 ? ROUNDS_BLOCK
                            : g->scale_mode == A8W8_SCALE_MX_E8M0_1x32 ? ROUNDS_MXFP8_ROWS : ROUNDS_PLAIN;
    if (c_tile_fits(g->stride_c, fp32 ? 4 : 2) && rounds_on_128_tiles(kind, g->m, g->n, g->k / BK, g->batch, fp32, num_cus(), g->b_preshuffled != 0)) return true;
    return fits_128_tiles(g->m, g->n, g->batch, num_cus());
}

// One variant of the 128-tile kernel: stages, tile columns, partial K steps, tile rows.
template <int MODE, int CDT, int STAGES, int BN_, bool RAGGED, int BM_>
int launch_tiles(const GemmParams& p, int batch, hipStream_t stream)
{
    GemmParams q = p;
    q.tiles_m = (p.m + BM_ - 1) / BM_;
    q.tiles_n = (p.n + BN_ - 1) / BN_;
    q.inv_per_group = tile_map_inverse(8 * q.tiles_n);
    q.inv_rem = tile_map_inverse(q.tiles_m % 8);
    q.runs = tiles_in_runs(q.tiles_m, q.tiles_n, p.k / BK, batch, BM_ > BN_, num_cus());
    const dim3 grid((unsigned)(q.tiles_m * q.tiles_n), 1, (unsigned)batch);
    return launch(gemm_a8w8_tile128<MODE, CDT, STAGES, BN_, RAGGED, BM_>, grid, dim3(SM_THREADS), small_lds_bytes(MODE, STAGES, BN_, BM_), stream, q);
}

// The tile shape and depth of staging are tile128_variant's.
template <int MODE, int CDT, bool RAGGED = false>
int launch_small(const GemmParams& p, int batch, hipStream_t stream)
{
    // (256 x 128 tiles leave rows past the end to the buffer descriptors: the 32-bit offsets of a whole tile must not wrap)
    const bool tall = MODE != MODE_BLOCK && !RAGGED && (p.m + 256ll) * p.lda + p.k < (1ll << 32) && (p.n + 128ll) * p.ldb + p.k < (1ll << 32);
    switch (tile128_variant(p.m, p.n, p.k, batch, tall, MODE == MODE_BF16 || MODE == MODE_F4T, num_cus(), MODE == MODE_BLOCK && CDT == C_FP32)) {
        case TILES_64x64: return launch_tiles<MODE, CDT, SHORT_STAGES, 64, RAGGED, 64>(p, batch, stream);
        case TILES_128x64:
            if (narrow_tiles_deep(p.m, p.n, p.k, RAGGED ? STEP_OTHER : MODE == MODE_BLOCK ? STEP_BLOCK
                                                 : MODE == MODE_TENSOR || MODE == MODE_ROWCOL || MODE == MODE_MXT || MODE == MODE_BF16 ? STEP_LIGHT : STEP_OTHER))
                return launch_tiles<MODE, CDT, narrow_deep_stages(MODE), 64, RAGGED, 128>(p, batch, stream);
            return launch_tiles<MODE, CDT, NARROW_STAGES, 64, RAGGED, 128>(p, batch, stream);
        case TILES_128_FOUR_STAGES: return launch_tiles<MODE, CDT, 4, 128, RAGGED, 128>(p, batch, stream);
        case TILES_256x128:
            if constexpr (MODE != MODE_BLOCK && !RAGGED) return launch_tiles<MODE, CDT, 3, 128, false, 256>(p, batch, stream);
            [[fallthrough]];
        default: return launch_tiles<MODE, CDT, 2, 128, RAGGED, 128>(p, batch, stream);
    }
}

template <int MODE, int CDT>
int launch_wide(const GemmParams& p, int batch, hipStream_t stream);

// Persistent pipelined kernel (eight waves): one workgroup per CU walks the (batch, tile) list.
template <int MODE, int CDT>
int launch_persist(const GemmParams& p, int batch, hipStream_t stream)
{
    // tiled MX scales exist on the four-wave kernel only (whatever passes persist_ok with them also passes wide_ok)
    if constexpr (MODE == MODE_MXT) return launch_wide<MODE, CDT>(p, batch, stream);
    else {
    if (!c_tile_fits(p.ldc, CDT == C_BF16 ? 2 : 4)) return A8W8_ERR_TOO_LARGE;
    PersistParams pp;
    pp.g = p;
    pp.batch = batch;
    pp.items = batch * p.tiles_m * p.tiles_n;
    pp.map = make_tile_map(p.tiles_m, p.tiles_n, items_in_runs(p.tiles_m, p.tiles_n, p.k / BK, batch, num_cus()));
    const int cus = num_cus();
    dim3 grid((unsigned)(pp.items < cus ? pp.items : cus), 1, 1);
    return launch(gemm_a8w8_persist<MODE, CDT>, grid, dim3(GEMM_THREADS), persist_lds_bytes(MODE), stream, pp);
    }
}

// Four-wave persistent kernel (one wave per SIMD, 128 x 128 per wave).
template <int MODE, int CDT>
int launch_wide(const GemmParams& p, int batch, hipStream_t stream)
{
    if constexpr (MODE != MODE_BLOCK) {
        if (!c_tile_fits(p.ldc, CDT == C_BF16 ? 2 : 4)) return A8W8_ERR_TOO_LARGE;
        PersistParams pp;
        pp.g = p;
        pp.batch = batch;
        pp.items = batch * p.tiles_m * p.tiles_n;
        pp.map = make_tile_map(p.tiles_m, p.tiles_n, items_in_runs(p.tiles_m, p.tiles_n, p.k / BK, batch, num_cus()));
        const int cus = num_cus();
        dim3 grid((unsigned)(pp.items < cus ? pp.items : cus), 1, 1);
        return launch(gemm_a8w8_wide<MODE, CDT>, grid, dim3(WIDE_THREADS), wide_lds_bytes(MODE), stream, pp);
    } else {
        return launch_persist<MODE, CDT>(p, batch, stream);
    }
}

template <int MODE, int CDT>
int launch_general(const GemmParams& p, int batch, hipStream_t stream)
{
    dim3 grid((unsigned)((p.n + 15) / 16), (unsigned)((p.m + 15) / 16), (unsigned)batch);
    return launch(gemm_a8w8_general<MODE, CDT>, grid, dim3(256), 0, stream, p);
}


#define A8W8_DISPATCH(FN, mode, cdt, ...)                                                   \
    switch ((mode) * 2 + (cdt)) {                                                           \
        case 0: return FN<MODE_TENSOR, C_BF16>(__VA_ARGS__);                                \
        case 1: return FN<MODE_TENSOR, C_FP32>(__VA_ARGS__);                                \
        case 2: return FN<MODE_ROWCOL, C_BF16>(__VA_ARGS__);                                \
        case 3: return FN<MODE_ROWCOL, C_FP32>(__VA_ARGS__);                                \
        case 4: return FN<MODE_BLOCK, C_BF16>(__VA_ARGS__);                                 \
        case 5: return FN<MODE_BLOCK, C_FP32>(__VA_ARGS__);                                 \
        case 6: return FN<MODE_MX, C_BF16>(__VA_ARGS__);                                    \
        case 7: return FN<MODE_MX, C_FP32>(__VA_ARGS__);                                    \
        case 8: return FN<MODE_MXT, C_BF16>(__VA_ARGS__);                                   \
        case 9: return FN<MODE_MXT, C_FP32>(__VA_ARGS__);                                   \
        default: return A8W8_ERR_BAD_MODE;                                                  \
    }

int dispatch_persist(const a8w8_gemm_args* g, const GemmParams& p, hipStream_t s)
{
    A8W8_DISPATCH(launch_persist, g->scale_mode, g->c_dtype, p, g->batch, s)
}
int dispatch_wide(const a8w8_gemm_args* g, const GemmParams& p, hipStream_t s)
{
    A8W8_DISPATCH(launch_wide, g->scale_mode, g->c_dtype, p, g->batch, s)
}
int dispatch_small(const a8w8_gemm_args* g, const GemmParams& p, hipStream_t s)
{
    A8W8_DISPATCH(launch_small, g->scale_mode, g->c_dtype, p, g->batch, s)
}
int dispatch_ragged(const a8w8_gemm_args* g, const GemmParams& p, hipStream_t s)
{
    if (g->scale_mode == A8W8_SCALE_TENSOR)
        return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_TENSOR, C_BF16, true>(p, g->batch, s) : launch_small<MODE_TENSOR, C_FP32, true>(p, g->batch, s);
    return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_ROWCOL, C_BF16, true>(p, g->batch, s) : launch_small<MODE_ROWCOL, C_FP32, true>(p, g->batch, s);
}
int dispatch_general(const a8w8_gemm_args* g, const GemmParams& p, hipStream_t s)
{
    A8W8_DISPATCH(launch_general, g->scale_mode, g->c_dtype, p, g->batch, s)
}

// The flat kernels take up to 128 activation rows: up to four groups of 16 share one pass over the weights, past
// 64 rows two workgroups per group of weight tiles make two passes (the second one from L2).
constexpr int FLAT_MAX_M = 128;

int validate_flat(const a8w8_gemm_args* g)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    if (!g->b_preshuffled) return A8W8_ERR_BAD_MODE;
    if (g->scale_mode != A8W8_SCALE_ROWCOL && g->scale_mode != A8W8_SCALE_TENSOR && g->scale_mode != A8W8_SCALE_MX_E8M0_TILED &&
        g->scale_mode != A8W8_SCALE_BLOCK_1x128_128x128)
        return A8W8_ERR_BAD_MODE;
    const int st = validate_common(g);
    if (st != A8W8_OK) return st;
    if (g->m > FLAT_MAX_M) return A8W8_ERR_BAD_SHAPE;
    if (g->n % 16 != 0 || g->k % 64 != 0) return A8W8_ERR_BAD_GROUP;
    if (!aligned16(g->a) || !aligned16(g->b) || g->stride_a % 16 != 0) return A8W8_ERR_MISALIGNED;
    if (g->batch > 1 && (g->stride_a_batch % 16 != 0 || g->stride_b_batch % 16 != 0)) return A8W8_ERR_MISALIGNED;
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_TILED &&
        (!aligned16(g->sfa) || !aligned16(g->sfb) || (g->batch > 1 && (g->stride_sfa_batch % 16 != 0 || g->stride_sfb_batch % 16 != 0))))
        return A8W8_ERR_MISALIGNED;
    return A8W8_OK;
}

template <int NT, int MT, int CDT, int MODE, bool BROW>
int launch_flat_nt(const GemmParams& p, int batch, hipStream_t stream)
{
    const int n_tiles = p.n / 16;
    dim3 grid((unsigned)(((n_tiles + NT - 1) / NT) * ((p.m + 16 * MT - 1) / (16 * MT))), 1, (unsigned)batch);
    return launch(flatmm_a8w8<NT, MT, CDT, MODE, BROW>, grid, dim3(FLAT_THREADS), 0, stream, p);
}

// The split of weight tiles and row groups is flat_split's.
template <int CDT, int MODE, bool BROW = false>
int launch_flat(const GemmParams& p, int batch, hipStream_t stream)
{
    constexpr FlatKind KIND = MODE == MODE_MXT ? FLAT_MXFP8 : MODE == MODE_F4T ? FLAT_MXFP4 : MODE == MODE_BLOCK ? FLAT_BLOCK
                              : MODE == MODE_BF16 ? FLAT_BF16 : FLAT_FP8;
    const FlatSplit split = flat_split(KIND, BROW, p.m, p.n, p.k, batch, num_cus());
    switch (10 * split.nt + split.mt) {
        case 11: return launch_flat_nt<1, 1, CDT, MODE, BROW>(p, batch, stream);
        case 12: return launch_flat_nt<1, 2, CDT, MODE, BROW>(p, batch, stream);
        case 21: return launch_flat_nt<2, 1, CDT, MODE, BROW>(p, batch, stream);
        case 22: return launch_flat_nt<2, 2, CDT, MODE, BROW>(p, batch, stream);
        case 23: return launch_flat_nt<2, 3, CDT, MODE, BROW>(p, batch, stream);
        case 24: return launch_flat_nt<2, 4, CDT, MODE, BROW>(p, batch, stream);
        case 26: return launch_flat_nt<2, 6, CDT, MODE, BROW>(p, batch, stream);
        case 41: return launch_flat_nt<4, 1, CDT, MODE, BROW>(p, batch, stream);
        case 42: return launch_flat_nt<4, 2, CDT, MODE, BROW>(p, batch, stream);
        case 43: return launch_flat_nt<4, 3, CDT, MODE, BROW>(p, batch, stream);
        case 44: return launch_flat_nt<4, 4, CDT, MODE, BROW>(p, batch, stream);
        default: return A8W8_ERR_BAD_MODE;
    }
}

// On shuffled weights both the flat GEMM and the MFMA kernels can run a skinny problem; the entry points take the one that the cost
// model of flat_is_faster calls faster.
// Row-major weights (a8w8_gemm without b_preshuffled; the flat kernel stages the weight rows through LDS, whole lines
// per load): as fast as shuffled ones unless the rows are a large power of two apart, where the 16 rows of a tile fall
// on the same memory channels -- 16384 x 7168 FP8 M = 16 / 32 / 64: 20 / 21 / 25 us, 8192 x 8192: 17 / 17 / 20 us
// (13 / 14 / 18 shuffled).
int g_route = A8W8_ROUTE_MODEL;      // a8w8_route_override

bool prefer_flat(int m, int n, long long row_bytes, int batch, double layout_factor = 1.0)
{
    if (g_route != A8W8_ROUTE_MODEL) return g_route == A8W8_ROUTE_FLAT;
    return flat_is_faster(m, n, row_bytes, batch, layout_factor, num_cus());
}

bool prefer_flat_fp8(const a8w8_gemm_args* g)
{
    const bool mx = g->scale_mode == A8W8_SCALE_MX_E8M0_TILED;
    const double layout_factor = g->b_preshuffled ? 1.0 : g->stride_b % 4096 == 0 ? 1.3 : 1.05;
    // (MXFP8 costs the flat kernel more than the dense one: 1.0, 1.05 and 1.1 fit the measured cells equally well)
    return prefer_flat(g->m, g->n, g->k, g->batch, layout_factor * (mx ? 1.1 : 1.0));
}

template <bool BROW>
int launch_flat_fp8_layout(const a8w8_gemm_args* g, hipStream_t s)
{
    const GemmParams p = make_params(g);
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_TILED)
        return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_MXT, BROW>(p, g->batch, s) : launch_flat<C_FP32, MODE_MXT, BROW>(p, g->batch, s);
    if (g->scale_mode == A8W8_SCALE_BLOCK_1x128_128x128)
        return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_BLOCK, BROW>(p, g->batch, s) : launch_flat<C_FP32, MODE_BLOCK, BROW>(p, g->batch, s);
    const bool tensor = g->scale_mode == A8W8_SCALE_TENSOR;
    if (g->c_dtype == A8W8_C_BF16)
        return tensor ? launch_flat<C_BF16, MODE_TENSOR, BROW>(p, g->batch, s) : launch_flat<C_BF16, MODE_ROWCOL, BROW>(p, g->batch, s);
    return tensor ? launch_flat<C_FP32, MODE_TENSOR, BROW>(p, g->batch, s) : launch_flat<C_FP32, MODE_ROWCOL, BROW>(p, g->batch, s);
}

int launch_flat_fp8(const a8w8_gemm_args* g, hipStream_t s)
{
    return g->b_preshuffled ? launch_flat_fp8_layout<false>(g, s) : launch_flat_fp8_layout<true>(g, s);
}

// A skinny problem on row-major weights that the flat kernel can run (it stages the weight rows through LDS).
bool flat_rowmajor_ok(const a8w8_gemm_args* g)
{
    if (g->b_preshuffled || g->m > FLAT_MAX_M) return false;
    if (g->scale_mode != A8W8_SCALE_ROWCOL && g->scale_mode != A8W8_SCALE_TENSOR && g->scale_mode != A8W8_SCALE_MX_E8M0_TILED &&
        g->scale_mode != A8W8_SCALE_BLOCK_1x128_128x128)
        return false;
    if (g->n % 16 != 0 || g->k % 64 != 0) return false;
    if (!aligned16(g->a) || !aligned16(g->b) || g->stride_a % 16 != 0 || g->stride_b % 16 != 0) return false;
    if (g->batch > 1 && (g->stride_a_batch % 16 != 0 || g->stride_b_batch % 16 != 0)) return false;
    if (g->scale_mode == A8W8_SCALE_MX_E8M0_TILED &&
        (!aligned16(g->sfa) || !aligned16(g->sfb) || (g->batch > 1 && (g->stride_sfa_batch % 16 != 0 || g->stride_sfb_batch % 16 != 0))))
        return false;
    return (long long)(g->n - 1) * g->stride_b + g->k < (1ll << 31);
}

// Whether launch_dense_fp8 (and the bf16 / MXFP4 entry points on their byte views) would take one of the two 256-tile
// kernels: their C tiles must fit 32-bit offsets (c_tile_fits), which the entry points check before any device call.
bool takes_tile256(const a8w8_gemm_args* g, bool fp4)
{
    return tiled_ok(g) && !small_ok(g, fp4) && persist_ok(g, fp4);
}
bool c_stride_too_large(const a8w8_gemm_args* g, const a8w8_gemm_args* byte_view, bool fp4 = false)
{
    return takes_tile256(byte_view, fp4) && !c_tile_fits(g->stride_c, g->c_dtype == A8W8_C_BF16 ? 2 : 4);
}

int launch_dense_fp8(const a8w8_gemm_args* g, hipStream_t s)
{
    const GemmParams p = make_params(g);
    if (ragged_ok(g)) return dispatch_ragged(g, p, s);
    if (!tiled_ok(g)) return dispatch_general(g, p, s);
    if (small_ok(g)) return dispatch_small(g, p, s);
    if (wide_ok(g)) return dispatch_wide(g, p, s);
    // what is left has a single K step (k = 128) or more work items than the persistent kernels index: the 128-tile
    // kernel runs any number of steps and tiles
    return persist_ok(g) ? dispatch_persist(g, p, s) : dispatch_small(g, p, s);
}

// the vectorised quantisers read 16 bytes per lane and write packed words
bool quant_vec_ok(const float* src, int rows, int k, int ld, const uint8_t* q, int q_align)
{
    return aligned16(src) && ld % 4 == 0 && k % 4 == 0 && ((uintptr_t)q & (uintptr_t)(q_align - 1)) == 0 &&
           (long long)rows * k < (1ll << 31);
}

// 127 at the positions of the tiled layout that no (row, block) owns, for quantisers that write the real ones only
int fill_mx_tiled(int rows, int k, uint8_t* scale, hipStream_t s)
{
    if (rows % 64 == 0 && k % 512 == 0) return A8W8_OK;
    const size_t dwords = mx_tiled_bytes(rows, k) / 4;
    return launch(mx_tiled_fill_kernel, dim3((unsigned)((dwords + 255) / 256)), dim3(256), 0, s, (uint32_t*)scale, dwords);
}

// The vectorised MX quantisers: row-major scales over the flattened array (quant_mx_flat_kernel); tiled ones by lines of the scales or as many chunks per
// wave as the array fills the chip with (quant_mx_lines_kernel, quant_mx_vec_kernel), over the padded array where mx_padding_in_launch says so.
template <bool FP4, bool TILED>
int launch_quant_mx(const float* src, int rows, int k, int ld, uint8_t* q, uint8_t* scale, hipStream_t s)
{
    if constexpr (!TILED) {
        const unsigned total = (unsigned)rows * (unsigned)k;
        const auto flat = [&](auto kernel, unsigned chunks) {
            return launch(kernel, dim3((total + 1024 * chunks - 1) / (1024 * chunks)), dim3(256), 0, s, src, total, (unsigned)k, (unsigned)ld, q, scale);
        };
        switch (quant_mx_chunks(FP4, total, ld != k)) {
            case 1: return flat(quant_mx_flat_kernel<FP4, 1>, 1);
            case 2: return flat(quant_mx_flat_kernel<FP4, 2>, 2);
            default: return flat(quant_mx_flat_kernel<FP4, 4>, 4);
        }
    } else {
        int rows_p = rows, k_p = k;
        if (mx_padding_in_launch(rows, k)) {
            rows_p = (rows + 63) / 64 * 64;
            k_p = (k + 511) / 512 * 512;
            const MxLines lines = quant_mx_by_lines(FP4, rows, k);
            if (lines != MX_NOT_BY_LINES) {
                const unsigned col_groups = (unsigned)(k_p / 256);
                return launch(lines == MX_LINES_FOUR_WAVES ? quant_mx_lines_kernel<FP4, 4> : quant_mx_lines_kernel<FP4, 8>, dim3((unsigned)(rows_p / 16) * col_groups),
                              dim3(lines == MX_LINES_FOUR_WAVES ? 256 : 512), 0, s, src, rows, k, ld, q, scale, col_groups);
            }
        } else if (const int st = fill_mx_tiled(rows, k, scale, s); st != A8W8_OK) {
            return st;
        }
        const long long total = (long long)rows_p * k_p;
        const auto grid = [&](int per_thread) { return dim3((unsigned)((total / per_thread + 255) / 256)); };
        if (total >= QUANT_MX_FULL) return launch(quant_mx_vec_kernel<FP4, 4>, grid(16), dim3(256), 0, s, src, rows, k, rows_p, k_p, ld, q, scale);
        if constexpr (FP4) {
            return launch(quant_mxfp4_few_kernel, grid(8), dim3(256), 0, s, src, rows, k, rows_p, k_p, ld, q, scale);
        } else {
            if (total > QUANT_MX_FEW) return launch(quant_mx_vec_kernel<false, 2>, grid(8), dim3(256), 0, s, src, rows, k, rows_p, k_p, ld, q, scale);
            return launch(quant_mx_vec_kernel<false, 1>, grid(4), dim3(256), 0, s, src, rows, k, rows_p, k_p, ld, q, scale);
        }
    }
}

}  // namespace

extern "C" {

int a8w8_gemm(const a8w8_gemm_args* args, void* hip_stream)
{
    const int st = validate_common(args);
    if (st != A8W8_OK) return st;
    a8w8_gemm_args local = *args;
    if (local.b_preshuffled) local.stride_b = local.k;      // stride_b is not read for shuffled weights
    const a8w8_gemm_args* g = &local;
    const int shuf = validate_shuffled_b(g);
    if (shuf != A8W8_OK) return shuf;
    // a skinny problem on shuffled weights: the flat kernel where it is the faster one
    const bool flat = (g->b_preshuffled && validate_flat(g) == A8W8_OK && prefer_flat_fp8(g)) || (flat_rowmajor_ok(g) && prefer_flat_fp8(g));
    if (!flat && c_stride_too_large(g, g)) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    if (flat) return launch_flat_fp8(g, s);
    return launch_dense_fp8(g, s);
}

static int a16w16_flat_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_dense);

static int a16w16_gemm_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_flat)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    // a skinny problem on shuffled weights: the flat kernel where it is the faster one (and can run it)
    if (allow_flat && g->b_preshuffled && g->m > 0 && g->m <= FLAT_MAX_M && prefer_flat(g->m, g->n, 2ll * g->k, g->batch) &&
        a16w16_flat_impl(g, hip_stream, false) == A8W8_OK)
        return A8W8_OK;
    if (!g->a || !g->b || !g->c) return A8W8_ERR_NULL_POINTER;
    if (g->m <= 0 || g->n <= 0 || g->k <= 0 || g->batch <= 0) return A8W8_ERR_BAD_SHAPE;
    if (g->c_dtype != A8W8_C_BF16 && g->c_dtype != A8W8_C_FP32) return A8W8_ERR_BAD_MODE;
    if (g->stride_c < g->n || g->stride_a < g->k || (!g->b_preshuffled && g->stride_b < g->k)) return A8W8_ERR_BAD_STRIDE;
    if (g->batch > 1 && (g->stride_a_batch < 0 || g->stride_b_batch < 0 || g->stride_c_batch < 0)) return A8W8_ERR_BAD_STRIDE;
    const long long a_span = ((long long)(g->m - 1) * g->stride_a + g->k) * 2;
    const long long b_span = (g->b_preshuffled ? (long long)g->n * g->k : (long long)(g->n - 1) * g->stride_b + g->k) * 2;
    if (a_span >= (1ll << 31) || b_span >= (1ll << 31) || g->batch > 65535) return A8W8_ERR_TOO_LARGE;
    // the tiled kernel reads bf16 rows as byte rows of 2k columns
    a8w8_gemm_args bytes = *g;
    bytes.k = g->k * 2;
    bytes.stride_a = g->stride_a * 2; bytes.stride_b = g->b_preshuffled ? bytes.k : g->stride_b * 2;
    bytes.stride_a_batch = g->stride_a_batch * 2; bytes.stride_b_batch = g->stride_b_batch * 2;
    bytes.scale_mode = A8W8_SCALE_TENSOR;
    const bool fits = (long long)g->stride_a_batch * 2 < (1ll << 31) && (long long)g->stride_b_batch * 2 < (1ll << 31);
    const bool flat_rows = fits && flat_rowmajor_ok(&bytes) && prefer_flat(g->m, g->n, bytes.k, g->batch, bytes.stride_b % 4096 == 0 ? 1.3 : 1.05);
    if (!flat_rows && fits && c_stride_too_large(g, &bytes)) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    // a skinny problem on row-major weights: the flat kernel (weight rows staged through LDS) where it is the faster one
    if (flat_rows) {
        GemmParams p = make_params(&bytes);
        p.sfa = p.sfb = nullptr;
        return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_BF16, true>(p, g->batch, s)
                                         : launch_flat<C_FP32, MODE_BF16, true>(p, g->batch, s);
    }
    // weights shuffled as bytes (a16w16_flatmm's): MFMA kernels only
    if (g->b_preshuffled && (validate_shuffled_b(&bytes) != A8W8_OK || !fits || !persist_ok(&bytes))) return A8W8_ERR_BAD_GROUP;
    if (fits && tiled_ok(&bytes) && persist_ok(&bytes)) {
        GemmParams p = make_params(&bytes);
        p.sfa = p.sfb = nullptr;
        if (small_ok(&bytes))            // few tiles: 128 x 128 ones
            return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_BF16, C_BF16>(p, g->batch, s)
                                             : launch_small<MODE_BF16, C_FP32>(p, g->batch, s);
        if (steps_on_four_waves(&bytes, false))
            return g->c_dtype == A8W8_C_BF16 ? launch_wide<MODE_BF16, C_BF16>(p, g->batch, s)
                                             : launch_wide<MODE_BF16, C_FP32>(p, g->batch, s);
        return g->c_dtype == A8W8_C_BF16 ? launch_persist<MODE_BF16, C_BF16>(p, g->batch, s)
                                         : launch_persist<MODE_BF16, C_FP32>(p, g->batch, s);
    }
    if (fits && ragged_ok(&bytes)) {     // a partial last K step
        GemmParams p = make_params(&bytes);
        p.sfa = p.sfb = nullptr;
        return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_BF16, C_BF16, true>(p, g->batch, s)
                                         : launch_small<MODE_BF16, C_FP32, true>(p, g->batch, s);
    }
    dim3 grid((unsigned)((g->n + 15) / 16), (unsigned)((g->m + 15) / 16), (unsigned)g->batch);
    if (g->c_dtype == A8W8_C_BF16)
        A8W8_LAUNCH_OR_RETURN((gemm_a16w16_general<C_BF16>), grid, dim3(256), 0, s, (const unsigned short*)g->a,
                           (const unsigned short*)g->b, g->c, g->m, g->n, g->k, g->stride_a, g->stride_b, g->stride_c,
                           (long long)g->stride_a_batch, (long long)g->stride_b_batch, (long long)g->stride_c_batch);
    else
        A8W8_LAUNCH_OR_RETURN((gemm_a16w16_general<C_FP32>), grid, dim3(256), 0, s, (const unsigned short*)g->a,
                           (const unsigned short*)g->b, g->c, g->m, g->n, g->k, g->stride_a, g->stride_b, g->stride_c,
                           (long long)g->stride_a_batch, (long long)g->stride_b_batch, (long long)g->stride_c_batch);
    return A8W8_OK;
}

int a16w16_gemm(const a8w8_gemm_args* g, void* hip_stream) { return a16w16_gemm_impl(g, hip_stream, true); }

static int a4w4_flat_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_dense);

static int a4w4_gemm_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_flat)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    // a skinny problem on shuffled weights: the flat kernel where it is the faster one (and can run it)
    if (allow_flat && g->b_preshuffled && g->m > 0 && g->m <= FLAT_MAX_M && prefer_flat(g->m, g->n, g->k / 2, g->batch) &&
        a4w4_flat_impl(g, hip_stream, false) == A8W8_OK)
        return A8W8_OK;
    if (!g->a || !g->b || !g->c || !g->sfa || !g->sfb) return A8W8_ERR_NULL_POINTER;
    if (g->m <= 0 || g->n <= 0 || g->k <= 0 || g->batch <= 0) return A8W8_ERR_BAD_SHAPE;
    if (g->scale_mode != A8W8_SCALE_MX_E8M0_1x32 && g->scale_mode != A8W8_SCALE_MX_E8M0_TILED) return A8W8_ERR_BAD_MODE;
    if (g->c_dtype != A8W8_C_BF16 && g->c_dtype != A8W8_C_FP32) return A8W8_ERR_BAD_MODE;
    if (g->k % 32 != 0) return A8W8_ERR_BAD_GROUP;
    if (g->stride_c < g->n || g->stride_a < g->k || (!g->b_preshuffled && g->stride_b < g->k)) return A8W8_ERR_BAD_STRIDE;
    if ((g->stride_a & 1) || (!g->b_preshuffled && (g->stride_b & 1))) return A8W8_ERR_MISALIGNED;      // rows start on a byte
    const bool tiled = g->scale_mode == A8W8_SCALE_MX_E8M0_TILED;
    if (!tiled && (g->stride_sfa < g->k / 32 || g->stride_sfb < g->k / 32)) return A8W8_ERR_BAD_STRIDE;
    if (g->batch > 1 && ((g->stride_a_batch & 1) || (g->stride_b_batch & 1))) return A8W8_ERR_MISALIGNED;
    if (g->batch > 1 && (g->stride_a_batch < 0 || g->stride_b_batch < 0 || g->stride_c_batch < 0 ||
                         g->stride_sfa_batch < 0 || g->stride_sfb_batch < 0))
        return A8W8_ERR_BAD_STRIDE;
    const long long a_span = ((long long)(g->m - 1) * g->stride_a + g->k) / 2;
    const long long b_span = (g->b_preshuffled ? (long long)g->n * g->k : (long long)(g->n - 1) * g->stride_b + g->k) / 2;
    if (a_span >= (1ll << 31) || b_span >= (1ll << 31) || g->batch > 65535) return A8W8_ERR_TOO_LARGE;
    // the tiled kernel reads packed rows as byte rows of k/2 columns
    a8w8_gemm_args bytes = *g;
    bytes.k = g->k / 2;
    bytes.stride_a = g->stride_a / 2; bytes.stride_b = g->b_preshuffled ? bytes.k : g->stride_b / 2;
    bytes.stride_a_batch = g->stride_a_batch / 2; bytes.stride_b_batch = g->stride_b_batch / 2;
    bytes.scale_mode = A8W8_SCALE_MX_E8M0_TILED;
    const bool flat_rows = tiled && flat_rowmajor_ok(&bytes) && prefer_flat(g->m, g->n, bytes.k, g->batch, bytes.stride_b % 4096 == 0 ? 1.3 : 1.05);
    if (!flat_rows && tiled && g->k % 256 == 0 && c_stride_too_large(g, &bytes, true)) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    // a skinny problem on row-major weights: the flat kernel where it is the faster one
    if (flat_rows) {
        const GemmParams p = make_params(&bytes);
        return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_F4T, true>(p, g->batch, s)
                                         : launch_flat<C_FP32, MODE_F4T, true>(p, g->batch, s);
    }
    // weights shuffled as bytes (a4w4_flatmm's): MFMA kernels only
    if (g->b_preshuffled && (!tiled || g->k % 256 != 0 || validate_shuffled_b(&bytes) != A8W8_OK ||
                             (!small_ok(&bytes, true) && !persist_ok(&bytes, true))))
        return A8W8_ERR_BAD_GROUP;
    // row-major scales: the 128-tile kernel at any size (it stages the step's eight scale bytes per row as two dwords:
    // scale rows have to start on dwords), the four-wave kernel where the problem fills the chip with 256-tiles and the
    // scale rows take its 16-byte loads
    if (!tiled && !g->b_preshuffled && g->k % 256 == 0) {
        a8w8_gemm_args rows = bytes;
        rows.scale_mode = A8W8_SCALE_MX_E8M0_1x32;      // what tiled_ok checks the scale strides and pointers against
        if (tiled_ok(&rows) && (long long)((g->m + SM_BM - 1) / SM_BM) * ((g->n + 63) / 64) < (1ll << 31)) {
            const GemmParams p = make_params(&bytes);
            if (wide_row_scales_ok(&rows))
                return g->c_dtype == A8W8_C_BF16 ? launch_wide<MODE_F4, C_BF16>(p, g->batch, s)
                                                 : launch_wide<MODE_F4, C_FP32>(p, g->batch, s);
            return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_F4, C_BF16>(p, g->batch, s)
                                             : launch_small<MODE_F4, C_FP32>(p, g->batch, s);
        }
    }
    if (tiled && g->k % 256 == 0 && tiled_ok(&bytes)) {
        const GemmParams p = make_params(&bytes);
        if (small_ok(&bytes, true))       // few tiles, or few K steps, an odd number
            return g->c_dtype == A8W8_C_BF16 ? launch_small<MODE_F4T, C_BF16>(p, g->batch, s)
                                             : launch_small<MODE_F4T, C_FP32>(p, g->batch, s);
        if (persist_ok(&bytes, true))
            return g->c_dtype == A8W8_C_BF16 ? launch_wide<MODE_F4T, C_BF16>(p, g->batch, s)
                                             : launch_wide<MODE_F4T, C_FP32>(p, g->batch, s);
    }
    dim3 grid((unsigned)((g->n + 15) / 16), (unsigned)((g->m + 15) / 16), (unsigned)g->batch);
#define A4W4_GENERAL(CDT, TILED)                                                                                        \
    A8W8_LAUNCH_OR_RETURN((gemm_a4w4_general<CDT, TILED>), grid, dim3(256), 0, s, (const uint8_t*)g->a, (const uint8_t*)g->b, \
                       (const uint8_t*)g->sfa, (const uint8_t*)g->sfb, g->c, g->m, g->n, g->k, g->stride_a / 2,            \
                       g->stride_b / 2, g->stride_c, g->stride_sfa, g->stride_sfb, (long long)g->stride_a_batch / 2,       \
                       (long long)g->stride_b_batch / 2, (long long)g->stride_c_batch, (long long)g->stride_sfa_batch,     \
                       (long long)g->stride_sfb_batch)
    if (g->c_dtype == A8W8_C_BF16) { if (tiled) A4W4_GENERAL(C_BF16, true); else A4W4_GENERAL(C_BF16, false); }
    else { if (tiled) A4W4_GENERAL(C_FP32, true); else A4W4_GENERAL(C_FP32, false); }
#undef A4W4_GENERAL
    return A8W8_OK;
}

int a4w4_gemm(const a8w8_gemm_args* g, void* hip_stream) { return a4w4_gemm_impl(g, hip_stream, true); }

static int a4w4_flat_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_dense)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    if (!g->a || !g->b || !g->c || !g->sfa || !g->sfb) return A8W8_ERR_NULL_POINTER;
    if (!g->b_preshuffled || g->scale_mode != A8W8_SCALE_MX_E8M0_TILED) return A8W8_ERR_BAD_MODE;
    if (g->m <= 0 || g->n <= 0 || g->k <= 0 || g->batch <= 0 || g->m > FLAT_MAX_M) return A8W8_ERR_BAD_SHAPE;
    if (g->c_dtype != A8W8_C_BF16 && g->c_dtype != A8W8_C_FP32) return A8W8_ERR_BAD_MODE;
    if (g->n % 16 != 0 || g->k % 128 != 0) return A8W8_ERR_BAD_GROUP;
    if (g->stride_c < g->n || g->stride_a < g->k) return A8W8_ERR_BAD_STRIDE;
    if (g->batch > 1 && (g->stride_a_batch < 0 || g->stride_b_batch < 0 || g->stride_c_batch < 0 ||
                         g->stride_sfa_batch < 0 || g->stride_sfb_batch < 0))
        return A8W8_ERR_BAD_STRIDE;
    if (!aligned16(g->a) || !aligned16(g->b) || !aligned16(g->sfa) || !aligned16(g->sfb) || g->stride_a % 32 != 0)
        return A8W8_ERR_MISALIGNED;
    if (g->batch > 1 && (g->stride_a_batch % 32 != 0 || g->stride_b_batch % 32 != 0 || g->stride_sfa_batch % 16 != 0 ||
                         g->stride_sfb_batch % 16 != 0))
        return A8W8_ERR_MISALIGNED;
    if ((long long)g->n * g->k / 2 >= (1ll << 31) || g->batch > 65535) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    // several groups of 16 rows over weights too large to stay in cache: the MFMA kernels read the same weights
    if (allow_dense && !prefer_flat(g->m, g->n, g->k / 2, g->batch) && a4w4_gemm_impl(g, hip_stream, false) == A8W8_OK)
        return A8W8_OK;
    a8w8_gemm_args bytes = *g;      // packed rows as byte rows of k/2 columns
    bytes.k = g->k / 2;
    bytes.stride_a = g->stride_a / 2; bytes.stride_b = g->k / 2;
    bytes.stride_a_batch = g->stride_a_batch / 2; bytes.stride_b_batch = g->stride_b_batch / 2;
    const GemmParams p = make_params(&bytes);
    hipStream_t s = (hipStream_t)hip_stream;
    return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_F4T>(p, g->batch, s) : launch_flat<C_FP32, MODE_F4T>(p, g->batch, s);
}

int a4w4_flatmm(const a8w8_gemm_args* g, void* hip_stream) { return a4w4_flat_impl(g, hip_stream, true); }

int a4w4_quantize_mx(const float* src, int rows, int k, int ld, uint8_t* q, uint8_t* scale, int tiled, void* hip_stream)
{
    if (!src || !q || !scale) return A8W8_ERR_NULL_POINTER;
    if (rows <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (k % 32 != 0) return A8W8_ERR_BAD_GROUP;
    if (ld < k) return A8W8_ERR_BAD_STRIDE;
    if (tiled && ((uintptr_t)scale & 3)) return A8W8_ERR_MISALIGNED;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    const long long threads = (long long)rows * k;
    if (quant_vec_ok(src, rows, k, ld, q, 4))
        return tiled ? launch_quant_mx<true, true>(src, rows, k, ld, q, scale, s) : launch_quant_mx<true, false>(src, rows, k, ld, q, scale, s);
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (!tiled) return launch(quant_mxfp4_kernel<false>, grid, dim3(256), 0, s, src, rows, k, ld, q, scale);
    if (const int st = fill_mx_tiled(rows, k, scale, s); st != A8W8_OK) return st;
    return launch(quant_mxfp4_kernel<true>, grid, dim3(256), 0, s, src, rows, k, ld, q, scale);
}

static int a16w16_flat_impl(const a8w8_gemm_args* g, void* hip_stream, bool allow_dense)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    if (!g->a || !g->b || !g->c) return A8W8_ERR_NULL_POINTER;
    if (!g->b_preshuffled) return A8W8_ERR_BAD_MODE;
    if (g->m <= 0 || g->n <= 0 || g->k <= 0 || g->batch <= 0 || g->m > FLAT_MAX_M) return A8W8_ERR_BAD_SHAPE;
    if (g->c_dtype != A8W8_C_BF16 && g->c_dtype != A8W8_C_FP32) return A8W8_ERR_BAD_MODE;
    if (g->n % 16 != 0 || g->k % 32 != 0) return A8W8_ERR_BAD_GROUP;
    if (g->stride_c < g->n || g->stride_a < g->k) return A8W8_ERR_BAD_STRIDE;
    if (!aligned16(g->a) || !aligned16(g->b) || g->stride_a % 8 != 0) return A8W8_ERR_MISALIGNED;
    if (g->batch > 1 && (g->stride_a_batch % 8 != 0 || g->stride_b_batch % 8 != 0)) return A8W8_ERR_MISALIGNED;
    if ((long long)g->n * g->k * 2 >= (1ll << 31) || g->batch > 65535) return A8W8_ERR_TOO_LARGE;
    // batch strides are doubled into byte counts held in an int
    if (g->batch > 1 && ((long long)g->stride_a_batch * 2 >= (1ll << 31) || (long long)g->stride_b_batch * 2 >= (1ll << 31)))
        return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    // several groups of 16 rows over weights too large to stay in cache: the MFMA kernels read the same weights
    if (allow_dense && !prefer_flat(g->m, g->n, 2ll * g->k, g->batch) && a16w16_gemm_impl(g, hip_stream, false) == A8W8_OK)
        return A8W8_OK;
    a8w8_gemm_args bytes = *g;      // bf16 rows as byte rows of 2k columns
    bytes.k = g->k * 2;
    bytes.stride_a = g->stride_a * 2; bytes.stride_b = g->k * 2;
    bytes.stride_a_batch = g->stride_a_batch * 2; bytes.stride_b_batch = g->stride_b_batch * 2;
    GemmParams p = make_params(&bytes);
    p.sfa = p.sfb = nullptr;
    hipStream_t s = (hipStream_t)hip_stream;
    return g->c_dtype == A8W8_C_BF16 ? launch_flat<C_BF16, MODE_BF16>(p, g->batch, s)
                                     : launch_flat<C_FP32, MODE_BF16>(p, g->batch, s);
}

int a16w16_flatmm(const a8w8_gemm_args* g, void* hip_stream) { return a16w16_flat_impl(g, hip_stream, true); }

int a8w8_gemm_blockscale(const a8w8_gemm_args* g, void* hip_stream)
{
    if (!g) return A8W8_ERR_NULL_POINTER;
    a8w8_gemm_args local = *g;
    local.scale_mode = A8W8_SCALE_BLOCK_1x128_128x128;
    return a8w8_gemm(&local, hip_stream);
}

int a8w8_flatmm(const a8w8_gemm_args* g, void* hip_stream)
{
    const int st = validate_flat(g);
    if (st != A8W8_OK) return st;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    // several groups of 16 rows over weights too large to stay in cache: the MFMA kernels read the same weights
    if (!prefer_flat_fp8(g)) {
        a8w8_gemm_args local = *g;
        local.stride_b = local.k;
        if (validate_shuffled_b(&local) == A8W8_OK) return launch_dense_fp8(&local, s);
    }
    return launch_flat_fp8(g, s);
}

static size_t shuffled_index(int j, int p, int k)
{
    return (((size_t)(j / 16) * (k / 64) + p / 64) * 4 + (p % 64) / 16) * 256 + (size_t)(j % 16) * 16 + p % 16;
}

int a8w8_preshuffle_b(const void* b_host, void* out_host, int n, int k)
{
    if (!b_host || !out_host) return A8W8_ERR_NULL_POINTER;
    if (n <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (n % 16 != 0 || k % 64 != 0) return A8W8_ERR_BAD_GROUP;
    const uint8_t* b = (const uint8_t*)b_host;
    uint8_t* o = (uint8_t*)out_host;
    for (int j = 0; j < n; ++j)
        for (int p = 0; p < k; p += 16) memcpy(o + shuffled_index(j, p, k), b + (size_t)j * k + p, 16);
    return A8W8_OK;
}

int a8w8_unshuffle_b(const void* bshuf_host, void* out_host, int n, int k)
{
    if (!bshuf_host || !out_host) return A8W8_ERR_NULL_POINTER;
    if (n <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (n % 16 != 0 || k % 64 != 0) return A8W8_ERR_BAD_GROUP;
    const uint8_t* s = (const uint8_t*)bshuf_host;
    uint8_t* o = (uint8_t*)out_host;
    for (int j = 0; j < n; ++j)
        for (int p = 0; p < k; p += 16) memcpy(o + (size_t)j * k + p, s + shuffled_index(j, p, k), 16);
    return A8W8_OK;
}

int a8w8_preshuffle_b_device(const void* b_dev, void* out_dev, int n, int k, void* hip_stream)
{
    if (!b_dev || !out_dev) return A8W8_ERR_NULL_POINTER;
    if (n <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (n % 16 != 0 || k % 64 != 0) return A8W8_ERR_BAD_GROUP;
    if (!aligned16(out_dev)) return A8W8_ERR_MISALIGNED;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    const long long units = (long long)n * k / 16;
    A8W8_LAUNCH_OR_RETURN(preshuffle_b_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0,
                       (hipStream_t)hip_stream, (const uint8_t*)b_dev, (uint8_t*)out_dev, n, k);
    return A8W8_OK;
}

int a8w8_cvt_f32_to_e4m3(const float* src, uint8_t* dst, size_t n, int dialect, int clamp240, void* hip_stream)
{
    if (dialect != A8W8_E4M3_OCP && dialect != A8W8_E4M3_FNUZ) return A8W8_ERR_BAD_MODE;
    if (n == 0) return A8W8_OK;
    if (!src || !dst) return A8W8_ERR_NULL_POINTER;
    if ((n + 3) / 4 > 0x7fffffffull * 256) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    const dim3 block(256);
    if (aligned16(src) && ((uintptr_t)dst & 3) == 0 && !(dialect == A8W8_E4M3_FNUZ && cvt_fnuz_few(n))) {
        const dim3 grid((unsigned)((n / 4 + 256 * CVT_UNITS) / (256 * CVT_UNITS)));      // (one thread at least, for the last n % 4)
        if (dialect == A8W8_E4M3_OCP)
            return clamp240 ? launch(cvt_f32_to_e4m3_vec_kernel<0, 1>, grid, block, 0, s, src, dst, n)
                            : launch(cvt_f32_to_e4m3_vec_kernel<0, 0>, grid, block, 0, s, src, dst, n);
        return clamp240 ? launch(cvt_f32_to_e4m3_vec_kernel<1, 1>, grid, block, 0, s, src, dst, n)
                        : launch(cvt_f32_to_e4m3_vec_kernel<1, 0>, grid, block, 0, s, src, dst, n);
    }
    const dim3 grid((unsigned)(((n + 3) / 4 + 255) / 256));
    if (dialect == A8W8_E4M3_OCP)
        return clamp240 ? launch(cvt_f32_to_e4m3_kernel<0, 1>, grid, block, 0, s, src, dst, n)
                        : launch(cvt_f32_to_e4m3_kernel<0, 0>, grid, block, 0, s, src, dst, n);
    return clamp240 ? launch(cvt_f32_to_e4m3_kernel<1, 1>, grid, block, 0, s, src, dst, n)
                    : launch(cvt_f32_to_e4m3_kernel<1, 0>, grid, block, 0, s, src, dst, n);
}

int a8w8_cvt_e4m3_to_f32(const uint8_t* src, float* dst, size_t n, int dialect, void* hip_stream)
{
    if (dialect != A8W8_E4M3_OCP && dialect != A8W8_E4M3_FNUZ) return A8W8_ERR_BAD_MODE;
    if (n == 0) return A8W8_OK;
    if (!src || !dst) return A8W8_ERR_NULL_POINTER;
    if (n > 0x7fffffffull * 256) return A8W8_ERR_TOO_LARGE;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    hipStream_t s = (hipStream_t)hip_stream;
    const dim3 block(256);
    if (((uintptr_t)src & 3) == 0 && aligned16(dst) && !(dialect == A8W8_E4M3_FNUZ && cvt_fnuz_few(n))) {
        const dim3 grid((unsigned)((n / 4 + 256 * CVT_UNITS) / (256 * CVT_UNITS)));
        return dialect == A8W8_E4M3_OCP ? launch(cvt_e4m3_to_f32_vec_kernel<0>, grid, block, 0, s, src, dst, n)
                                        : launch(cvt_e4m3_to_f32_vec_kernel<1>, grid, block, 0, s, src, dst, n);
    }
    const dim3 grid((unsigned)((n + 255) / 256));
    return dialect == A8W8_E4M3_OCP ? launch(cvt_e4m3_to_f32_kernel<0>, grid, block, 0, s, src, dst, n)
                                    : launch(cvt_e4m3_to_f32_kernel<1>, grid, block, 0, s, src, dst, n);
}

int a8w8_quantize(const float* src, int rows, int k, int ld, uint8_t* q, void* scale, int scale_mode, int group_rows,
                  void* hip_stream)
{
    return a8w8_quantize_ws(src, rows, k, ld, q, scale, scale_mode, group_rows, nullptr, 0, hip_stream);
}

size_t a8w8_quantize_workspace_bytes(int rows, int k, int scale_mode)
{
    return scale_mode == A8W8_SCALE_TENSOR && rows > 0 && k > 0 && (long long)rows * k > 4ll * QUANT_TENSOR_ONE ? sizeof(float) * QUANT_TENSOR_WS_PARTS : 0;
}

int a8w8_quantize_ws(const float* src, int rows, int k, int ld, uint8_t* q, void* scale, int scale_mode, int group_rows, void* workspace,
                     size_t workspace_bytes, void* hip_stream)
{
    if (!src || !q || !scale) return A8W8_ERR_NULL_POINTER;
    if (rows <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (ld < k) return A8W8_ERR_BAD_STRIDE;
    hipStream_t s = (hipStream_t)hip_stream;
    switch (scale_mode) {
        case A8W8_SCALE_TENSOR: {
            if (const int ds = device_status(); ds != A8W8_OK) return ds;
            const long long total = (long long)rows * k;
            if (ld == k && total % 4 == 0 && aligned16(src) && ((uintptr_t)q & 3) == 0) {
                const size_t units = (size_t)(total / 4);
                if (units <= QUANT_TENSOR_ONE)
                    return launch(quant_tensor_one_kernel, dim3(1), dim3(1024), 0, s, (const float4*)src, (int)units, (uint32_t*)q, (float*)scale);
                const unsigned parts = (unsigned)std::min<size_t>((units + 1023) / 1024, QUANT_TENSOR_PARTS);
                const size_t apply = (units + 256 * QUANT_TENSOR_UNITS - 1) / (256 * QUANT_TENSOR_UNITS);
                // (a launch has less than 2^32 threads along a dimension; the kernels below walk an array of any size with a fixed grid)
                if (apply * 256 < (1ull << 32)) {
                    if (workspace && aligned16(workspace) && workspace_bytes >= sizeof(float) * QUANT_TENSOR_WS_PARTS) {
                        const unsigned few = ((unsigned)std::min<size_t>((units + 1023) / 1024, QUANT_TENSOR_WS_PARTS) + 3) / 4 * 4;
                        A8W8_LAUNCH_OR_RETURN(quant_tensor_amax_ws_kernel, dim3(few), dim3(512), 0, s, (const float4*)src, units, (float*)workspace);
                        return launch(quant_tensor_apply_ws_kernel, dim3((unsigned)apply), dim3(256), 0, s, (const float4*)src, units, (uint32_t*)q, (float*)scale,
                                      (const float*)workspace, (int)few);
                    }
                    A8W8_LAUNCH_OR_RETURN(quant_tensor_amax_vec_kernel, dim3(parts), dim3(256), 0, s, (const float4*)src, units, (float*)q);
                    A8W8_LAUNCH_OR_RETURN(quant_tensor_fold_kernel, dim3(1), dim3(256), 0, s, (const float*)q, (int)parts, (float*)scale);
                    return launch(quant_tensor_apply_vec_kernel, dim3((unsigned)apply), dim3(256), 0, s, (const float4*)src, units, (uint32_t*)q,
                                  (const float*)scale);
                }
            }
            const unsigned grid = (unsigned)(total / 256 + 1 < 4096 ? total / 256 + 1 : 4096);
            A8W8_LAUNCH_OR_RETURN(quant_tensor_clear_kernel, dim3(1), dim3(1), 0, s, (float*)scale);
            A8W8_LAUNCH_OR_RETURN(quant_tensor_amax_kernel, dim3(grid), dim3(256), 0, s, src, rows, k, ld, (float*)scale);
            A8W8_LAUNCH_OR_RETURN(quant_tensor_apply_kernel, dim3(grid), dim3(256), 0, s, src, rows, k, ld, q, (const float*)scale);
            return launch(quant_tensor_finish_kernel, dim3(1), dim3(1), 0, s, (float*)scale);
        }
        case A8W8_SCALE_ROWCOL:
            if (const int ds = device_status(); ds != A8W8_OK) return ds;
            if (quant_vec_ok(src, rows, k, ld, q, 4) && quant_rows_by_wave(rows, k))
                return launch(quant_rowwise_wave_kernel, dim3((unsigned)((rows + 3ll) / 4)), dim3(256), 0, s, src, rows, k, ld, q, (float*)scale);
            if (quant_vec_ok(src, rows, k, ld, q, 4))
                return launch(k <= 4096 ? quant_rowwise_vec_kernel<256, true> : k <= 8192 ? quant_rowwise_vec_kernel<512, true>
                              : k <= 16384 ? quant_rowwise_vec_kernel<1024, true> : quant_rowwise_vec_kernel<256, false>,
                              dim3((unsigned)rows), dim3(k <= 4096 || k > 16384 ? 256 : k <= 8192 ? 512 : 1024), 0, s, src, k, ld, q, (float*)scale);
            else
                A8W8_LAUNCH_OR_RETURN(quant_rowwise_kernel, dim3((unsigned)rows), dim3(256), 0, s, src, k, ld, q, (float*)scale);
            return A8W8_OK;
        case A8W8_SCALE_BLOCK_1x128_128x128:
            if (k % 128 != 0) return A8W8_ERR_BAD_GROUP;
            if (group_rows == 1) {
                if (const int ds = device_status(); ds != A8W8_OK) return ds;
                const long long waves = (long long)rows * (k / 128);
                const unsigned groups = (unsigned)(k / 128);
                if (quant_vec_ok(src, rows, k, ld, q, 4) && quant_1x128_along_rows(rows, k))
                    return waves > QUANT_1X128_FEW ? launch(quant_1x128_along_rows_kernel<4>, dim3((unsigned)((waves + 31) / 32)), dim3(256), 0, s, src,
                                                            rows, k, ld, q, (float*)scale)
                                                   : launch(quant_1x128_along_rows_kernel<1>, dim3((unsigned)((waves + 7) / 8)), dim3(256), 0, s, src,
                                                            rows, k, ld, q, (float*)scale);
                if (quant_vec_ok(src, rows, k, ld, q, 4) && (waves <= QUANT_1X128_FEW || rows < 32))
                    A8W8_LAUNCH_OR_RETURN(quant_1x128_vec_kernel<8>, dim3(groups * ((rows + 7) / 8)), dim3(256), 0, s, src, rows, k, ld, q,
                                       (float*)scale);
                else if (quant_vec_ok(src, rows, k, ld, q, 4))
                    A8W8_LAUNCH_OR_RETURN(quant_1x128_vec_kernel<32>, dim3(groups * ((rows + 31) / 32)), dim3(256), 0, s, src, rows, k, ld, q,
                                       (float*)scale);
                else
                    A8W8_LAUNCH_OR_RETURN(quant_1x128_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, src, rows, k,
                                       ld, q, (float*)scale);
                return A8W8_OK;
            }
            if (group_rows == 128) {
                if (rows % 128 != 0) return A8W8_ERR_BAD_GROUP;
                if (const int ds = device_status(); ds != A8W8_OK) return ds;
                if (quant_vec_ok(src, rows, k, ld, q, 4))
                    A8W8_LAUNCH_OR_RETURN(quant_128x128_vec_kernel, dim3((unsigned)(k / 128), (unsigned)(rows / 128)), dim3(256), 0,
                                       s, src, k, ld, q, (float*)scale);
                else
                    A8W8_LAUNCH_OR_RETURN(quant_128x128_kernel, dim3((unsigned)(k / 128), (unsigned)(rows / 128)), dim3(256), 0,
                                       s, src, k, ld, q, (float*)scale);
                return A8W8_OK;
            }
            return A8W8_ERR_BAD_MODE;
        case A8W8_SCALE_MX_E8M0_1x32: {
            if (k % 32 != 0) return A8W8_ERR_BAD_GROUP;
            if (const int ds = device_status(); ds != A8W8_OK) return ds;
            if (quant_vec_ok(src, rows, k, ld, q, 4)) return launch_quant_mx<false, false>(src, rows, k, ld, q, (uint8_t*)scale, s);
            return launch(quant_mx_kernel<false>, dim3((unsigned)(((long long)rows * k + 255) / 256)), dim3(256), 0, s, src, rows, k, ld, q,
                          (uint8_t*)scale);
        }
        case A8W8_SCALE_MX_E8M0_TILED: {
            if (k % 32 != 0) return A8W8_ERR_BAD_GROUP;
            if (const int ds = device_status(); ds != A8W8_OK) return ds;
            if (((uintptr_t)scale & 3) != 0) return A8W8_ERR_MISALIGNED;
            if (quant_vec_ok(src, rows, k, ld, q, 4)) return launch_quant_mx<false, true>(src, rows, k, ld, q, (uint8_t*)scale, s);
            if (const int st = fill_mx_tiled(rows, k, (uint8_t*)scale, s); st != A8W8_OK) return st;
            return launch(quant_mx_kernel<true>, dim3((unsigned)(((long long)rows * k + 255) / 256)), dim3(256), 0, s, src, rows, k, ld, q,
                          (uint8_t*)scale);
        }
        default:
            return A8W8_ERR_BAD_MODE;
    }
}

int a8w8_mx_tile_scales(const uint8_t* sf, int rows, int k, int stride, uint8_t* out, void* hip_stream)
{
    if (!sf || !out) return A8W8_ERR_NULL_POINTER;
    if (rows <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (k % 32 != 0) return A8W8_ERR_BAD_GROUP;
    if (stride < k / 32) return A8W8_ERR_BAD_STRIDE;
    if (!aligned16(out)) return A8W8_ERR_MISALIGNED;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    const size_t units = mx_tiled_bytes(rows, k) >> 10;
    A8W8_LAUNCH_OR_RETURN(mx_tile_scales_kernel, dim3((unsigned)((units + 3) / 4)), dim3(256), 0,
                       (hipStream_t)hip_stream, sf, rows, stride, out, (const uint8_t*)nullptr, 0, 0, (uint8_t*)nullptr, k);
    return A8W8_OK;
}

int a8w8_mx_tile_scales_ab(const uint8_t* sfa, int m, int stride_sfa, uint8_t* out_a, const uint8_t* sfb, int n,
                           int stride_sfb, uint8_t* out_b, int k, void* hip_stream)
{
    if (!sfa || !out_a || !sfb || !out_b) return A8W8_ERR_NULL_POINTER;
    if (m <= 0 || n <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (k % 32 != 0) return A8W8_ERR_BAD_GROUP;
    if (stride_sfa < k / 32 || stride_sfb < k / 32) return A8W8_ERR_BAD_STRIDE;
    if (!aligned16(out_a) || !aligned16(out_b)) return A8W8_ERR_MISALIGNED;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    const size_t units0 = mx_tiled_bytes(m, k) >> 10, units1 = mx_tiled_bytes(n, k) >> 10;
    A8W8_LAUNCH_OR_RETURN(mx_tile_scales_kernel, dim3((unsigned)((units0 + units1 + 3) / 4)), dim3(256), 0,
                       (hipStream_t)hip_stream, sfa, m, stride_sfa, out_a, sfb, n, stride_sfb, out_b, k);
    return A8W8_OK;
}

size_t a8w8_mx_tiled_bytes(int rows, int k)
{
    if (rows <= 0 || k <= 0) return 0;
    return mx_tiled_bytes(rows, k);
}

// ------------------------------------------------------------ weight files (host only)
namespace {
const char kWeightMagic[8] = {'A', '8', 'W', '8', 'W', 'G', 'T', 0};

uint64_t fnv1a64(const void* data, size_t n, uint64_t h)
{
    const uint8_t* p = (const uint8_t*)data;
    for (size_t i = 0; i < n; ++i) { h ^= p[i]; h *= 1099511628211ull; }
    return h;
}

int check_header(const a8w8_weight_header& h)
{
    if (memcmp(h.magic, kWeightMagic, 8) != 0 || h.version != 1) return A8W8_ERR_BAD_FILE;
    if (h.n == 0 || h.k == 0 || h.n > (1u << 30) || h.k > (1u << 30)) return A8W8_ERR_BAD_FILE;
    if (h.b_bytes != (uint64_t)h.n * h.k) return A8W8_ERR_BAD_FILE;
    if (h.scale_bytes == 0 || h.scale_bytes != a8w8_weight_scale_bytes((int)h.n, (int)h.k, (int)h.scale_mode))
        return A8W8_ERR_BAD_FILE;
    return A8W8_OK;
}
}  // namespace

size_t a8w8_weight_scale_bytes(int n, int k, int scale_mode)
{
    if (n <= 0 || k <= 0) return 0;
    switch (scale_mode) {
        case A8W8_SCALE_TENSOR: return 4;
        case A8W8_SCALE_ROWCOL: return (size_t)n * 4;
        case A8W8_SCALE_BLOCK_1x128_128x128: return (n % 128 || k % 128) ? 0 : (size_t)(n / 128) * (k / 128) * 4;
        case A8W8_SCALE_MX_E8M0_1x32: return k % 32 ? 0 : (size_t)n * (k / 32);
        case A8W8_SCALE_MX_E8M0_TILED: return k % 32 ? 0 : mx_tiled_bytes(n, k);
        default: return 0;
    }
}

int a8w8_weights_save(const char* path, const void* b_host, const void* scale_host, int n, int k, int b_preshuffled,
                      int scale_mode)
{
    if (!path || !b_host || !scale_host) return A8W8_ERR_NULL_POINTER;
    if (n <= 0 || k <= 0) return A8W8_ERR_BAD_SHAPE;
    if (b_preshuffled && (n % 16 != 0 || k % 64 != 0)) return A8W8_ERR_BAD_GROUP;
    const size_t sbytes = a8w8_weight_scale_bytes(n, k, scale_mode);
    if (sbytes == 0) return scale_mode < 0 || scale_mode > A8W8_SCALE_MX_E8M0_TILED ? A8W8_ERR_BAD_MODE : A8W8_ERR_BAD_GROUP;
    a8w8_weight_header h;
    memset(&h, 0, sizeof h);
    memcpy(h.magic, kWeightMagic, 8);
    h.version = 1;
    h.n = (uint32_t)n; h.k = (uint32_t)k;
    h.b_preshuffled = b_preshuffled ? 1 : 0;
    h.scale_mode = (uint32_t)scale_mode;
    h.b_bytes = (uint64_t)n * k;
    h.scale_bytes = sbytes;
    h.checksum = fnv1a64(scale_host, sbytes, fnv1a64(b_host, (size_t)h.b_bytes, 14695981039346656037ull));
    FILE* f = fopen(path, "wb");
    if (!f) return A8W8_ERR_IO;
    const bool ok = fwrite(&h, sizeof h, 1, f) == 1 && fwrite(b_host, 1, (size_t)h.b_bytes, f) == h.b_bytes &&
                    fwrite(scale_host, 1, sbytes, f) == sbytes;
    return (fclose(f) == 0 && ok) ? A8W8_OK : A8W8_ERR_IO;
}

int a8w8_weights_info(const char* path, a8w8_weight_header* out)
{
    if (!path || !out) return A8W8_ERR_NULL_POINTER;
    FILE* f = fopen(path, "rb");
    if (!f) return A8W8_ERR_IO;
    const size_t got = fread(out, 1, sizeof *out, f);
    fclose(f);
    if (got != sizeof *out) return A8W8_ERR_BAD_FILE;
    return check_header(*out);
}

int a8w8_weights_load(const char* path, void* b_host, size_t b_capacity, void* scale_host, size_t scale_capacity)
{
    if (!path || !b_host || !scale_host) return A8W8_ERR_NULL_POINTER;
    FILE* f = fopen(path, "rb");
    if (!f) return A8W8_ERR_IO;
    a8w8_weight_header h;
    int st = fread(&h, 1, sizeof h, f) == sizeof h ? check_header(h) : A8W8_ERR_BAD_FILE;
    if (st == A8W8_OK && (h.b_bytes > b_capacity || h.scale_bytes > scale_capacity)) st = A8W8_ERR_BAD_STRIDE;
    if (st == A8W8_OK && (fread(b_host, 1, (size_t)h.b_bytes, f) != h.b_bytes ||
                          fread(scale_host, 1, (size_t)h.scale_bytes, f) != h.scale_bytes))
        st = A8W8_ERR_BAD_FILE;
    fclose(f);
    if (st != A8W8_OK) return st;
    const uint64_t sum = fnv1a64(scale_host, (size_t)h.scale_bytes, fnv1a64(b_host, (size_t)h.b_bytes, 14695981039346656037ull));
    return sum == h.checksum ? A8W8_OK : A8W8_ERR_BAD_FILE;
}

const char* a8w8_status_string(int status)
{
    switch (status) {
        case A8W8_OK: return "ok";
        case A8W8_ERR_NULL_POINTER: return "null pointer";
        case A8W8_ERR_BAD_SHAPE: return "m, n, k and batch must be positive (and m <= 128 for the flat GEMMs)";
        case A8W8_ERR_BAD_GROUP: return "m/n/k must be multiples of the scale group (or of the shuffle tile)";
        case A8W8_ERR_BAD_STRIDE: return "a stride is smaller than the extent it spans";
        case A8W8_ERR_MISALIGNED: return "pointer or stride not 16-byte aligned";
        case A8W8_ERR_BAD_MODE: return "unsupported scale mode, output type or layout flag";
        case A8W8_ERR_TOO_LARGE: return "matrix too large for 32-bit offsets";
        case A8W8_ERR_LAUNCH: return "kernel launch failed";
        case A8W8_ERR_NO_DEVICE: return "current device is not gfx950";
        case A8W8_ERR_IO: return "weight file could not be opened, read or written";
        case A8W8_ERR_BAD_FILE: return "not a weight file of this version, truncated, or checksum mismatch";
        default: return "unknown status";
    }
}

const char* a8w8_kernel_name(const a8w8_gemm_args* g)
{
    if (!g) return nullptr;
    // shuffled weights: a8w8_gemm and a8w8_flatmm both pick the flat kernel for skinny problems it runs faster
    a8w8_gemm_args local = *g;
    if (local.b_preshuffled) local.stride_b = local.k;
    g = &local;
    const bool dense_ok = validate_common(g) == A8W8_OK && validate_shuffled_b(g) == A8W8_OK;
    if (g->b_preshuffled && validate_flat(g) == A8W8_OK && (prefer_flat_fp8(g) || !dense_ok)) return "flatmm_a8w8";
    if (dense_ok && flat_rowmajor_ok(g) && prefer_flat_fp8(g)) return "flatmm_a8w8";
    if (!dense_ok) return nullptr;
    if (ragged_ok(g)) return "gemm_a8w8_tile128";
    if (!tiled_ok(g)) return "gemm_a8w8_general";
    if (small_ok(g)) return "gemm_a8w8_tile128";
    if (wide_ok(g)) return "gemm_a8w8_wide";
    return persist_ok(g) ? "gemm_a8w8_persist" : "gemm_a8w8_tile128";
}

int a8w8_hbm_read_probe(const void* src, size_t bytes, void* sink, void* hip_stream)
{
    if (!src || !sink) return A8W8_ERR_NULL_POINTER;
    if (bytes == 0) return A8W8_ERR_BAD_SHAPE;
    if (bytes % 16 != 0 || !aligned16(src) || ((uintptr_t)sink & 3)) return A8W8_ERR_MISALIGNED;
    if (const int ds = device_status(); ds != A8W8_OK) return ds;
    const size_t n16 = bytes / 16;
    // eight workgroups per compute unit (the best of the grids tried on a 117 MB buffer), fewer for buffers that do not
    // give every thread a load
    const size_t want = (n16 + HBM_PROBE_THREADS - 1) / HBM_PROBE_THREADS;
    const size_t most = (size_t)num_cus() * 8;
    const unsigned grid = (unsigned)(want < most ? want : most);
    return launch(hbm_read_probe_kernel, dim3(grid), dim3(HBM_PROBE_THREADS), 0, (hipStream_t)hip_stream, (const v4i*)src, n16,
                  (int*)sink);
}

int a8w8_route_override(int choice)
{
    if (choice != A8W8_ROUTE_MODEL && choice != A8W8_ROUTE_FLAT && choice != A8W8_ROUTE_DENSE) return A8W8_ERR_BAD_MODE;
    const int before = g_route;
    g_route = choice;
    return before;
}

int a8w8_init(int device)
{
    int current = 0;
    if (hipGetDevice(&current) != hipSuccess) return A8W8_ERR_NO_DEVICE;
    if (device < 0) device = current;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || device >= count || device >= MAX_DEVICES) return A8W8_ERR_NO_DEVICE;
    if (device != current && hipSetDevice(device) != hipSuccess) {
        (void)hipGetLastError();      // the failed switch must not linger as the thread's last error
        return A8W8_ERR_NO_DEVICE;
    }
    const int st = device_status();
    if (device != current) (void)hipSetDevice(current);
    return st;
}

// An ablated build (measurement switches of gemm_wide.hpp) reports a negative version, so that nothing mistakes it
// for the library.
int a8w8_version(void) { return A8W8_ABLATED ? -300 : 300; }

}  // extern "C"
