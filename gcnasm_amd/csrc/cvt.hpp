// fp8 <-> fp32 conversion helpers, weight pre-shuffle and the quantisation front end (gfx950).
#pragma once
#include "a8w8_device.hpp"

namespace a8w8 {

// ---------------------------------------------------------------- software E4M3 FNUZ
// The gfx942 dialect (bias 8, max 240, 0x80 = NaN, no -0) is not what gfx950 hardware
// converts to, so it is computed with integer arithmetic on the fp32 bit pattern.
A8W8_DEV uint8_t f32_to_e4m3_fnuz_sw(float x)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const uint32_t sign = (u >> 31) << 7;
    const uint32_t au = u & 0x7fffffffu;
    if (au >= 0x7f800000u) return 0x80;                 // NaN and Inf have one code
    if (au > 0x43700000u) return (uint8_t)(sign | 0x7f); // beyond 240: largest finite
    const int e8 = (int)(au >> 23) - 127 + 8;           // exponent field in the fp8 format
    uint32_t mant = au & 0x7fffffu;
    uint32_t code, rem, half;
    if (e8 >= 1) {
        code = ((uint32_t)e8 << 3) | (mant >> 20);
        rem = mant & 0xfffffu;
        half = 0x80000u;
    } else {
        const int sh = 21 - e8;                          // 20 dropped bits + (1 - e8)
        if (sh > 25) return 0;                           // below half of the smallest subnormal
        mant |= 0x800000u;
        code = mant >> sh;
        rem = mant & ((1u << sh) - 1u);
        half = 1u << (sh - 1);
    }
    if (rem > half || (rem == half && (code & 1u))) ++code;   // nearest, ties to even
    if (code > 0x7fu) code = 0x7fu;
    if (code == 0) return 0;
    return (uint8_t)(sign | code);
}

A8W8_DEV float e4m3_fnuz_to_f32_sw(uint8_t c)
{
    if (c == 0) return 0.f;
    if (c == 0x80) return __builtin_bit_cast(float, 0x7F800001u);
    uint32_t sign = (uint32_t)(c >> 7) << 31;
    int e = (c >> 3) & 15;
    uint32_t m = c & 7;
    if (e == 0) {                       // subnormal: shift the leading one into place
        const int lz = __builtin_clz(m) - 29;   // 0 for m>=4, 1 for m>=2, 2 for m==1
        m = (m << (lz + 1)) & 7;
        e = -lz;
    }
    return __builtin_bit_cast(float, sign | ((uint32_t)(e + 127 - 8) << 23) | (m << 20));
}

// to_fp8_raw_from_fp32 of the reference (cvt_fp8/test.cpp:21-43) on this hardware.
A8W8_DEV float clamp240_unless_special(float v)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    if ((u & 0x7F800000u) != 0x7F800000u) v = __builtin_amdgcn_fmed3f(v, 240.0f, -240.0f);
    return v;
}

// Four floats -> one packed word: two packed hardware converts into the low halves, merged by a byte permute
// (the sequence of pk_cvt_fp8x4_fp32x4_rne, pk_cvt/test.cpp:220-257).
template <int DIALECT, int CLAMP>
A8W8_DEV uint32_t cvt_four_to_e4m3(float a, float b, float c, float d)
{
    if (CLAMP) {
        a = clamp240_unless_special(a);
        b = clamp240_unless_special(b);
        c = clamp240_unless_special(c);
        d = clamp240_unless_special(d);
    }
    if (DIALECT == 0) {
        const uint32_t x = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
        const uint32_t y = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, 0, false);
        return __builtin_amdgcn_perm(y, x, 0x05040100);
    }
    return (uint32_t)f32_to_e4m3_fnuz_sw(a) | ((uint32_t)f32_to_e4m3_fnuz_sw(b) << 8) | ((uint32_t)f32_to_e4m3_fnuz_sw(c) << 16) |
           ((uint32_t)f32_to_e4m3_fnuz_sw(d) << 24);
}

// One thread converts four consecutive floats (decode: one code): arrays that do not start on 16 bytes (floats) or 4 bytes (codes),
// and FNUZ arrays that do not fill the chip (cvt_fnuz_few of routes.hpp).
template <int DIALECT, int CLAMP>
__global__ void __launch_bounds__(256) cvt_f32_to_e4m3_kernel(const float* src, uint8_t* dst, size_t n)
{
    const size_t i0 = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i0 >= n) return;
    float s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = i0 + e < n ? src[i0 + e] : 0.f;
    const uint32_t word = cvt_four_to_e4m3<DIALECT, CLAMP>(s[0], s[1], s[2], s[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (i0 + e < n) dst[i0 + e] = (uint8_t)(word >> (8 * e));
}

template <int DIALECT>
__global__ void __launch_bounds__(256) cvt_e4m3_to_f32_kernel(const uint8_t* src, float* dst, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint8_t c = src[i];
    dst[i] = DIALECT == 0 ? __builtin_amdgcn_cvt_f32_fp8((int)c, 0) : e4m3_fnuz_to_f32_sw(c);
}

// The same conversions of aligned arrays (bound: HBM, 5 bytes per element).  A thread takes CVT_UNITS groups of four
// elements 256 groups apart: every load and store of a wave covers one contiguous run, 16 bytes of floats and 4 of codes per
// lane, all loads before the first convert.  The floats, read or written once, go non-temporally, the codes, a fifth of the
// bytes, do not (a reader of fresh codes finds them in cache).  The last n % 4 elements fall to one thread.
// 4096 x 8192 values, encode / decode, us: 36 / 41 as one thread per four floats (scalar loads) or per code; 27.2 / 24.0 here
// (6.2 / 7.0 TB/s); floats with ordinary accesses 30.9 / 32.8; codes non-temporal as well 27.3 / 28.9; four groups per thread
// 27.8 / 24.6, eight 29.1 / 25.4, one 31.0 / 23.8.
constexpr int CVT_UNITS = 2;
template <int DIALECT, int CLAMP>
__global__ void __launch_bounds__(256) cvt_f32_to_e4m3_vec_kernel(const float* __restrict__ src, uint8_t* __restrict__ dst, size_t n)
{
    const size_t groups = n >> 2, u0 = (size_t)blockIdx.x * (256 * CVT_UNITS) + threadIdx.x;
    v4f v[CVT_UNITS];
#pragma unroll
    for (int u = 0; u < CVT_UNITS; ++u)
        if (u0 + 256 * u < groups) v[u] = __builtin_nontemporal_load((const v4f*)src + u0 + 256 * u);
#pragma unroll
    for (int u = 0; u < CVT_UNITS; ++u)
        if (u0 + 256 * u < groups)
            ((uint32_t*)dst)[u0 + 256 * u] = cvt_four_to_e4m3<DIALECT, CLAMP>(v[u].x, v[u].y, v[u].z, v[u].w);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) {
        for (size_t i = groups * 4; i < n; ++i) dst[i] = (uint8_t)cvt_four_to_e4m3<DIALECT, CLAMP>(src[i], 0.f, 0.f, 0.f);
    }
}

template <int DIALECT>
A8W8_DEV v4f cvt_four_to_f32(uint32_t w)
{
    if (DIALECT == 0)
        return v4f{__builtin_amdgcn_cvt_f32_fp8((int)w, 0), __builtin_amdgcn_cvt_f32_fp8((int)w, 1),
                   __builtin_amdgcn_cvt_f32_fp8((int)w, 2), __builtin_amdgcn_cvt_f32_fp8((int)w, 3)};
    return v4f{e4m3_fnuz_to_f32_sw((uint8_t)w), e4m3_fnuz_to_f32_sw((uint8_t)(w >> 8)), e4m3_fnuz_to_f32_sw((uint8_t)(w >> 16)),
               e4m3_fnuz_to_f32_sw((uint8_t)(w >> 24))};
}
template <int DIALECT>
__global__ void __launch_bounds__(256) cvt_e4m3_to_f32_vec_kernel(const uint8_t* __restrict__ src, float* __restrict__ dst, size_t n)
{
    const size_t groups = n >> 2, u0 = (size_t)blockIdx.x * (256 * CVT_UNITS) + threadIdx.x;
    uint32_t w[CVT_UNITS];
#pragma unroll
    for (int u = 0; u < CVT_UNITS; ++u)
        if (u0 + 256 * u < groups) w[u] = ((const uint32_t*)src)[u0 + 256 * u];
#pragma unroll
    for (int u = 0; u < CVT_UNITS; ++u)
        if (u0 + 256 * u < groups) __builtin_nontemporal_store(cvt_four_to_f32<DIALECT>(w[u]), (v4f*)dst + u0 + 256 * u);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) {
        for (size_t i = groups * 4; i < n; ++i) dst[i] = cvt_four_to_f32<DIALECT>(src[i]).x;
    }
}

// Row-major B[n][k] -> Bshuf[n/16][k/64][4][16][16 B]; one thread moves 16 bytes.
__global__ void __launch_bounds__(256) preshuffle_b_kernel(const uint8_t* b, uint8_t* out, int n, int k)
{
    const long long o = (long long)blockIdx.x * 256 + threadIdx.x;   // 16-byte unit in the output
    const long long total = (long long)n * k / 16;
    if (o >= total) return;
    const int r = (int)(o & 15);
    const int kq = (int)((o >> 4) & 3);
    const long long blk = o >> 6;
    const int k_tiles = k >> 6;
    const int kt = (int)(blk % k_tiles);
    const int nt = (int)(blk / k_tiles);
    const uint8_t* src = b + (long long)(nt * 16 + r) * k + kt * 64 + kq * 16;
    v4i v;
    if (((uintptr_t)src & 15) == 0) v = *(const v4i*)src;
    else __builtin_memcpy(&v, src, 16);
    *(v4i*)(out + o * 16) = v;
}

// ------------------------------------------------------------ quantisation front end
A8W8_DEV float wave_max(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

A8W8_DEV uint8_t quant_one(float x, float scale)
{
    const float q = __fdiv_rn(x, scale);
    const uint32_t w = __builtin_amdgcn_cvt_pk_fp8_f32(q, q, 0, false);
    return (uint8_t)w;
}

// per-row scale = amax(row)/448; one workgroup per row
__global__ void __launch_bounds__(256) quant_rowwise_kernel(const float* src, int k, int ld, uint8_t* q, float* scale)
{
    __shared__ float part[4];
    const int row = blockIdx.x;
    const float* x = src + (long long)row * ld;
    float amax = 0.f;
    for (int i = threadIdx.x; i < k; i += 256) amax = fmaxf(amax, fabsf(x[i]));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (threadIdx.x == 0) scale[row] = s;
    for (int i = threadIdx.x; i < k; i += 256) q[(long long)row * k + i] = quant_one(x[i], s);
}

// per-tensor scale = amax(all)/448 in three steps over the caller's one-float scale slot: clear it, fold
// every workgroup's |x| maximum into it (non-negative floats order like their bit patterns), quantise with
// amax/448, and finally turn the slot from amax into the scale.
__global__ void quant_tensor_clear_kernel(float* scale) { *scale = 0.f; }
__global__ void __launch_bounds__(256) quant_tensor_amax_kernel(const float* src, int rows, int k, int ld, float* scale)
{
    __shared__ float part[4];
    const long long total = (long long)rows * k;
    float amax = 0.f;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256)
        amax = fmaxf(amax, fabsf(src[(i / k) * ld + i % k]));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
        amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
        atomicMax((unsigned int*)scale, __float_as_uint(amax));
    }
}
__global__ void __launch_bounds__(256) quant_tensor_apply_kernel(const float* src, int rows, int k, int ld, uint8_t* q,
                                                                 const float* amax_slot)
{
    const long long total = (long long)rows * k;
    const float amax = *amax_slot;
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256)
        q[i] = quant_one(src[(i / k) * ld + i % k], s);
}
__global__ void quant_tensor_finish_kernel(float* scale)
{
    const float amax = *scale;
    *scale = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;
}

// 1 x 128 blocks: one wave per (row, 128-group); scale stored [k/128][rows]
__global__ void __launch_bounds__(256) quant_1x128_kernel(const float* src, int rows, int k, int ld, uint8_t* q,
                                                          float* scale)
{
    const int groups = k >> 7;
    const long long w = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= (long long)rows * groups) return;
    const int row = (int)(w / groups), g = (int)(w % groups);
    const int lane = threadIdx.x & 63;
    const float* x = src + (long long)row * ld + g * 128;
    const float v0 = x[lane], v1 = x[lane + 64];
    const float amax = wave_max(fmaxf(fabsf(v0), fabsf(v1)));
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (lane == 0) scale[(long long)g * rows + row] = s;
    uint8_t* o = q + (long long)row * k + g * 128;
    o[lane] = quant_one(v0, s);
    o[lane + 64] = quant_one(v1, s);
}

// 128 x 128 blocks: one workgroup per block; scale stored [rows/128][k/128]
__global__ void __launch_bounds__(256) quant_128x128_kernel(const float* src, int k, int ld, uint8_t* q, float* scale)
{
    __shared__ float part[4];
    const int gk = blockIdx.x, gr = blockIdx.y;
    const float* x = src + (long long)gr * 128 * ld + gk * 128;
    float amax = 0.f;
    for (int i = threadIdx.x; i < 128 * 128; i += 256) amax = fmaxf(amax, fabsf(x[(long long)(i >> 7) * ld + (i & 127)]));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (threadIdx.x == 0) scale[(long long)gr * gridDim.x + gk] = s;
    uint8_t* o = q + (long long)gr * 128 * k + gk * 128;
    for (int i = threadIdx.x; i < 128 * 128; i += 256)
        o[(long long)(i >> 7) * k + (i & 127)] = quant_one(x[(long long)(i >> 7) * ld + (i & 127)], s);
}

// clamp(ceil(log2(amax / top)), -127, 127) for top = (1 + TOP_MANT / 2^23) 2^TOP_EXP: the exponent difference, one more when
// amax's mantissa is above top's.  It equals the exponent of the rounded fp32 quotient for every amax: the quotient of the first
// mantissa above top's rounds up, except where it is subnormal, once (TOP_MANT + 1 at quotient exponent -127), where it rounds
// back to the power of two; amax = Inf keeps the exponent 0 that frexp gave it, NaN counts as zero.  Five integer operations
// where the divide and frexp took about twenty.
template <int TOP_EXP, unsigned TOP_MANT>
A8W8_DEV int mx_block_exponent(float amax)
{
    const unsigned u = __float_as_uint(amax);
    const int field = (int)(u >> 23);
    const unsigned above = (u & 0x7fffffu) > TOP_MANT + (field == TOP_EXP ? 1u : 0u) ? 1u : 0u;
    const int e = max(-127, field - 127 - TOP_EXP + (int)above);
    return u < 0x7f800000u ? e : u == 0x7f800000u ? 0 : -127;
}
A8W8_DEV int mx_exponent_e4m3(float amax) { return mx_block_exponent<8, 0x600000u>(amax); }      // 448 = 1.75 * 2^8
A8W8_DEV int mx_exponent_e2m1(float amax) { return mx_block_exponent<2, 0x400000u>(amax); }      // 6 = 1.5 * 2^2

// MX: one E8M0 exponent per 32 K-elements, e = ceil(log2(amax/448)) clamped to [-127, 127]; 32 lanes per block.
template <bool TILED>
__global__ void __launch_bounds__(256) quant_mx_kernel(const float* src, int rows, int k, int ld, uint8_t* q,
                                                       uint8_t* scale)
{
    const int blocks = k >> 5;
    const long long idx = ((long long)blockIdx.x * 256 + threadIdx.x) >> 5;
    if (idx >= (long long)rows * blocks) return;
    const int row = (int)(idx / blocks), g = (int)(idx % blocks);
    const int l = threadIdx.x & 31;
    const float v = src[(long long)row * ld + g * 32 + l];
    float amax = fabsf(v);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    const int e = mx_exponent_e4m3(amax);
    if (l == 0) scale[TILED ? mx_tiled_index(rows, row, g) : (size_t)row * blocks + g] = (uint8_t)(e + 127);
    const float qv = ldexpf(v, -e);
    const uint32_t w = __builtin_amdgcn_cvt_pk_fp8_f32(qv, qv, 0, false);
    q[(long long)row * k + g * 32 + l] = (uint8_t)w;
}

// natural [rows][k/32] E8M0 scales (row stride `stride` bytes) -> the tiled layout of mx_tiled_index.
// One thread per output dword: two tiles x two K steps of one (64-row block, r16, g, jp).
// Consecutive threads write consecutive dwords.  Rows past `rows` and blocks past k get 127
// (scale 1.0; their products are never formed or never stored).
// MXFP4: one E8M0 exponent per 32 K-elements, e = ceil(log2(amax/6)) clamped to [-127, 127]; elements
// become E2M1 (round to nearest, ties to the even mantissa bit, saturating at 6), two per byte with
// the even K index in the low nibble.  32 lanes per block; even lanes write the byte.
A8W8_DEV unsigned e2m1_encode(float x)
{
    const float a = fabsf(x);
    const unsigned code = (a > 0.25f) + (a >= 0.75f) + (a > 1.25f) + (a >= 1.75f) + (a > 2.5f) + (a >= 3.5f) + (a > 5.0f);
    return ((__float_as_uint(x) >> 31) << 3) | (a != a ? 7u : code);
}
template <bool TILED>
__global__ void __launch_bounds__(256) quant_mxfp4_kernel(const float* src, int rows, int k, int ld, uint8_t* q,
                                                          uint8_t* scale)
{
    const int blocks = k >> 5;
    const long long idx = ((long long)blockIdx.x * 256 + threadIdx.x) >> 5;
    if (idx >= (long long)rows * blocks) return;
    const int row = (int)(idx / blocks), g = (int)(idx % blocks);
    const int l = threadIdx.x & 31;
    const float v = src[(long long)row * ld + g * 32 + l];
    float amax = fabsf(v);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    const int e = mx_exponent_e2m1(amax);
    if (l == 0) scale[TILED ? mx_tiled_index(rows, row, g) : (size_t)row * blocks + g] = (uint8_t)(e + 127);
    const unsigned code = e2m1_encode(ldexpf(v, -e));
    const unsigned hi = __shfl_down(code, 1, 64);
    if ((l & 1) == 0) q[(long long)row * (k >> 1) + ((g * 32 + l) >> 1)] = (uint8_t)(code | (hi << 4));
}

// ------------------------------------------------------------ vectorised quantisers
// The kernels above move one element per thread (4-byte loads, 1-byte stores).  When rows are
// 16-byte aligned (src, ld % 4 == 0, k % 4 == 0) the kernels below do the same arithmetic on four
// elements per thread per chunk: 16-byte loads, one packed store, same bits out.
A8W8_DEV uint32_t pack4_e4m3(float a, float b, float c, float d)
{
    uint32_t w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    return __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
}
// two floats, divided by 2^e, as E2M1 codes in byte BYTE of `word`: the hardware convert, the same code as e2m1_encode(ldexpf(x, -e))
// for all 2^32 inputs (NaN and Inf included) at every e tried, -127 and 127 among them
template <int BYTE>
A8W8_DEV unsigned e2m1_pair(unsigned word, float x, float y, float scale)
{
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, x, y, scale, BYTE);
}

// 16 bytes of an input that is read once: a non-temporal load (the line is not kept in L2 in place of something that
// will be read again; 8192 x 8192 fp32 to FP8 with row scales 58.9 -> 54.2 us, to MXFP8 56.6 -> 54.1 us)
A8W8_DEV float4 load_once4(const float* p)
{
    const v4f t = __builtin_nontemporal_load((const v4f*)p);
    return make_float4(t.x, t.y, t.z, t.w);
}

// MX formats with one E8M0 exponent per 32 elements, tiled scales that do not leave by lines (bound: HBM).  A wave takes 256 CHUNKS consecutive elements of the
// flattened [rows, k] array: lane l owns elements 4l..4l+3 of each chunk of 256, eight lanes share a block.  Every load and
// store instruction of a wave covers one contiguous run of memory; all loads are issued before any chunk is processed.
// Four chunks are what large arrays want (8192 x 8192 E4M3, tiled scales: 56.3 us, two 58.3, one 64.9), fewer where there are
// not enough of them to fill the chip and a wave's own latency is the time (2560 x 2560: 8.2 / 7.4 / 8.5; 64 x 7168: 3.8 / 2.7 /
// 2.7; 16 x 7168: 3.7 / 2.6 / 2.3).  Tiled scales of arrays past a million elements: quant_mx_lines_kernel below; row-major ones: quant_mx_flat_kernel.
// The grid covers the padded [rows_p, k_p] array of the tiled layout (rows_p % 64 == 0, k_p % 512 == 0), so that the
// positions no (row, block) owns get their 127 here instead of from a launch of their own before this one (2.3 us).  Where that
// launch precedes this one (much padding: mx_padding_in_launch of routes.hpp), rows_p = rows and k_p = k.
// FP4: packed E2M1, two bytes per lane and chunk; the hardware convert instead of seven comparisons per element (8192 x 8192
// 62.6 -> 50.3 us, 4096 x 4096 16.8 -> 13.6).
template <bool FP4, int CHUNKS>
__global__ void __launch_bounds__(256) quant_mx_vec_kernel(const float* __restrict__ src, int rows, int k, int rows_p, int k_p, int ld,
                                                           uint8_t* __restrict__ q, uint8_t* __restrict__ scale)
{
    const unsigned total = (unsigned)rows_p * (unsigned)k_p;        // < 2^31 (checked by the host)
    const unsigned wave = (blockIdx.x * 256u + threadIdx.x) >> 6;
    const unsigned lane = threadIdx.x & 63;
    unsigned row[CHUNKS], col[CHUNKS];
    bool live[CHUNKS], owned[CHUNKS];
    float4 v[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const unsigned e0 = wave * (256u * CHUNKS) + c * 256u + lane * 4u;
        live[c] = e0 < total;
        row[c] = live[c] ? e0 / (unsigned)k_p : 0u;
        col[c] = live[c] ? e0 % (unsigned)k_p : 0u;
        owned[c] = live[c] && row[c] < (unsigned)rows && col[c] < (unsigned)k;
        v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (owned[c]) v[c] = load_once4(src + (size_t)row[c] * ld + col[c]);
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        float amax = fmaxf(fmaxf(fabsf(v[c].x), fabsf(v[c].y)), fmaxf(fabsf(v[c].z), fabsf(v[c].w)));
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const int e = FP4 ? mx_exponent_e2m1(amax) : mx_exponent_e4m3(amax);
        if (!live[c]) continue;
        if ((lane & 7) == 0) scale[mx_tiled_index(rows, (int)row[c], (int)(col[c] >> 5))] = (uint8_t)((owned[c] ? e : 0) + 127);
        if (!owned[c]) continue;
        if constexpr (FP4) {
            const float s = __uint_as_float((unsigned)(e + 127) << 23);      // (2^-127: the convert takes the exponent field)
            *(uint16_t*)(q + (((size_t)row[c] * k + col[c]) >> 1)) = (uint16_t)e2m1_pair<1>(e2m1_pair<0>(0u, v[c].x, v[c].y, s), v[c].z, v[c].w, s);
        } else {
            *(uint32_t*)(q + (size_t)row[c] * k + col[c]) =
                pack4_e4m3(ldexpf(v[c].x, -e), ldexpf(v[c].y, -e), ldexpf(v[c].z, -e), ldexpf(v[c].w, -e));
        }
    }
}

// MXFP4 with tiled scales below the size that fills the chip: lane l owns eight consecutive elements (two 16-byte loads, one 4-byte store), four
// lanes share a block, a wave takes 512 consecutive elements (256 x 8192: 2.7 us against 3.2-3.8 with chunks, 64 x 7168: 2.3
// against 2.6; 4096 x 2048: 7.8 against 7.5).
__global__ void __launch_bounds__(256) quant_mxfp4_few_kernel(const float* __restrict__ src, int rows, int k, int rows_p, int k_p, int ld,
                                                              uint8_t* __restrict__ q, uint8_t* __restrict__ scale)
{
    const unsigned total = (unsigned)rows_p * (unsigned)k_p;        // < 2^31 (checked by the host)
    const unsigned e0 = (blockIdx.x * 256u + threadIdx.x) * 8u;
    const bool live = e0 < total;
    const unsigned row = live ? e0 / (unsigned)k_p : 0u, col = live ? e0 % (unsigned)k_p : 0u;
    const bool owned = live && row < (unsigned)rows && col < (unsigned)k;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (owned) {
        const float* p = src + (size_t)row * ld + col;
        a = load_once4(p);
        b = load_once4(p + 4);
    }
    float amax = fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                       fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fmaxf(fabsf(b.z), fabsf(b.w))));
#pragma unroll
    for (int off = 2; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    const int e = mx_exponent_e2m1(amax);
    if (!live) return;
    if ((threadIdx.x & 3) == 0) scale[mx_tiled_index(rows, (int)row, (int)(col >> 5))] = (uint8_t)((owned ? e : 0) + 127);
    if (!owned) return;
    const float s = __uint_as_float((unsigned)(e + 127) << 23);
    *(uint32_t*)(q + (((size_t)row * k + col) >> 1)) =
        e2m1_pair<3>(e2m1_pair<2>(e2m1_pair<1>(e2m1_pair<0>(0u, a.x, a.y, s), a.z, a.w, s), b.x, b.y, s), b.z, b.w, s);
}

// The same for row-major scales (bound: HBM).  Codes and scales then lie as the flattened array does, code and block numbers are the element's own, and
// no row or column is computed unless the rows of the input are apart (ld != k): the divisions of quant_mx_vec_kernel stood before every load.  Two
// chunks per wave for whole arrays, four for rows apart, one where there are too few to fill the chip (quant_mx_chunks of routes.hpp).  us, rows and
// columns / flattened, E4M3, MXFP4: 8192 x 8192 54.5 -> 52.3, 50.8 -> 47.9 (6.0 TB/s), 4096 x 4096 16.5 -> 15.5, 14.6 -> 13.7, 2560 x 2560 7.6 -> 7.3,
// 7.5 -> 6.9, 300 x 5632 3.9 -> 3.2, 3.6 -> 3.5.  Scale bytes gathered into lines in LDS first: 0.1 to 0.4 us longer.
template <bool FP4, int CHUNKS>
__global__ void __launch_bounds__(256) quant_mx_flat_kernel(const float* __restrict__ src, unsigned total, unsigned k, unsigned ld, uint8_t* __restrict__ q,
                                                            uint8_t* __restrict__ scale)
{
    const unsigned lane = threadIdx.x & 63;
    const unsigned first = ((blockIdx.x * 256u + threadIdx.x) >> 6) * (256u * CHUNKS) + lane * 4u;      // (total < 2^31, checked by the host)
    float4 v[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const unsigned e0 = first + c * 256u;
        v[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e0 < total) v[c] = load_once4(src + (ld == k ? (size_t)e0 : (size_t)(e0 / k) * ld + e0 % k));
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const unsigned e0 = first + c * 256u;
        float amax = fmaxf(fmaxf(fabsf(v[c].x), fabsf(v[c].y)), fmaxf(fabsf(v[c].z), fabsf(v[c].w)));
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const int e = FP4 ? mx_exponent_e2m1(amax) : mx_exponent_e4m3(amax);
        if (e0 >= total) continue;
        if ((lane & 7) == 0) scale[e0 >> 5] = (uint8_t)(e + 127);
        if constexpr (FP4) {
            const float s = __uint_as_float((unsigned)(e + 127) << 23);
            *(uint16_t*)(q + (e0 >> 1)) = (uint16_t)e2m1_pair<1>(e2m1_pair<0>(0u, v[c].x, v[c].y, s), v[c].z, v[c].w, s);
        } else {
            *(uint32_t*)(q + e0) = pack4_e4m3(ldexpf(v[c].x, -e), ldexpf(v[c].y, -e), ldexpf(v[c].z, -e), ldexpf(v[c].w, -e));
        }
    }
}

// The same for tiled scales, by lines of the scale array (bound: HBM).  A workgroup takes the 16 rows and 256 columns whose scales are one
// 128-byte line of the tiled layout (rows 8x .. 8x + 7 and 32 + 8x .. of a 64-row block, one "pair"), a wave 16 / WAVES of the rows, 256
// columns per load; the scale bytes meet in LDS and leave as the line.  Written straight from the blocks, as above, they are single bytes of lines
// that a dozen workgroups on several L2s share.  Padding, rows and columns alike, is in the lines (127) and costs no element.
// us, E4M3 / MXFP4, above -> here: 8192 x 8192 55.8 -> 50.0 / 52.7 -> 45.7 (6.7 TB/s), 4096 x 4096 17.2 -> 15.0 / 16.2 -> 13.3, 5248 x 2688 15.8 -> 14.1 /
// 15.1 -> 13.0, 2560 x 2560 8.2 -> 7.4 / 7.5 -> 6.8, 256 x 8192 4.2 -> 3.9 / 3.8 -> 3.7 (of which a launch is 2.4).
// Four waves a workgroup between 5 and 15 million elements, eight otherwise (us, four / eight: 1012 x 4096 5.5 / 5.0, 3000 x 2048 6.8 / 7.0, 5831 x 2304 12.9 / 14.1,
// 4200 x 4096 15.8 / 15.3, 8192 x 4096 27.8 / 26.5).
template <bool FP4, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) quant_mx_lines_kernel(const float* __restrict__ src, int rows, int k, int ld, uint8_t* __restrict__ q,
                                                                    uint8_t* __restrict__ scale, unsigned col_groups)
{
    constexpr int R = 16 / WAVES;
    __shared__ __attribute__((aligned(16))) uint8_t line[128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cg = (int)(blockIdx.x % col_groups), rg = (int)(blockIdx.x / col_groups);      // 256 columns; block rg / 4, x = rg % 4
    const int col = cg * 256 + lane * 4;
    const bool col_owned = col < k;
    int row[R];
    float4 v[R];
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int r = wave * R + u;      // row r & 7 of the lower eight, or of the upper ones
        row[u] = (rg >> 2) * 64 + (rg & 3) * 8 + (r & 7) + (r >> 3) * 32;
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (col_owned && row[u] < rows) v[u] = load_once4(src + (size_t)row[u] * ld + col);
    }
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int r = wave * R + u;
        const bool owned = col_owned && row[u] < rows;
        float amax = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
#pragma unroll
        for (int off = 4; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const int e = FP4 ? mx_exponent_e2m1(amax) : mx_exponent_e4m3(amax);
        // (mx_tiled_index within the line: y = row % 4, g = block % 4, jp = upper eight, par = row / 4 % 2, s = block / 4)
        if ((lane & 7) == 0) line[((r & 3) * 4 + ((lane >> 3) & 3)) * 8 + (r >> 3) * 4 + ((r >> 2) & 1) * 2 + (lane >> 5)] = (uint8_t)((owned ? e : 0) + 127);
        if (!owned) continue;
        if constexpr (FP4) {
            const float s = __uint_as_float((unsigned)(e + 127) << 23);
            *(uint16_t*)(q + (((size_t)row[u] * k + col) >> 1)) = (uint16_t)e2m1_pair<1>(e2m1_pair<0>(0u, v[u].x, v[u].y, s), v[u].z, v[u].w, s);
        } else {
            *(uint32_t*)(q + (size_t)row[u] * k + col) =
                pack4_e4m3(ldexpf(v[u].x, -e), ldexpf(v[u].y, -e), ldexpf(v[u].z, -e), ldexpf(v[u].w, -e));
        }
    }
    __syncthreads();
    // (the array is on a dword at least)
    if (threadIdx.x < 32) {
        const size_t at = (((size_t)(cg >> 1) * ((rows + 63) >> 6) + (rg >> 2)) * 2 + (cg & 1)) * 512 + (rg & 3) * 128;
        ((uint32_t*)(scale + at))[threadIdx.x] = ((const uint32_t*)line)[threadIdx.x];
    }
}

// tiled scales: elements from which the chip is full; elements up to which a chunk per wave is the fastest (64 x 7168 3.3 us with two, 3.1 with one)
constexpr long long QUANT_MX_FULL = 1ll << 23, QUANT_MX_FEW = 1ll << 20;

// per-row scale, one workgroup per row.  HOLD: the row (at most 16 THREADS elements) stays in registers between the amax pass
// and the quantisation, four 16-byte loads per thread (one read of the input); otherwise it is read twice.  256 threads up to
// 4096 elements, 512 to 8192, 1024 to 16384: fewer registers and a shorter chain per thread than 256 threads with eight loads
// each (8192 x 8192 54.2 -> 52.0 us, 256 x 8192 4.2 -> 4.0, 16 x 7168 3.4 -> 3.2, 4096 x 2048 9.1 -> 8.5); more threads
// than that idle (4096 x 4096 15.2 us with 256, 17.8 with 512).
template <int THREADS, bool HOLD>
__global__ void __launch_bounds__(THREADS) quant_rowwise_vec_kernel(const float* __restrict__ src, int k, int ld,
                                                                    uint8_t* __restrict__ q, float* __restrict__ scale)
{
    __shared__ float part[THREADS / 64];
    const int row = blockIdx.x;
    const float* x = src + (size_t)row * ld;
    float4 held[4];
    float amax = 0.f;
    if constexpr (HOLD) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = threadIdx.x * 4 + u * (4 * THREADS);
            held[u] = i < k ? load_once4(x + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(held[u].x), fabsf(held[u].y)), fmaxf(fabsf(held[u].z), fabsf(held[u].w))));
    } else {
        for (int i = threadIdx.x * 4; i < k; i += 4 * THREADS) {
            const float4 v = *(const float4*)(x + i);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    }
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = part[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) amax = fmaxf(amax, part[w]);
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (threadIdx.x == 0) scale[row] = s;
    if constexpr (HOLD) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = threadIdx.x * 4 + u * (4 * THREADS);
            if (i < k)
                *(uint32_t*)(q + (size_t)row * k + i) = pack4_e4m3(__fdiv_rn(held[u].x, s), __fdiv_rn(held[u].y, s),
                                                                   __fdiv_rn(held[u].z, s), __fdiv_rn(held[u].w, s));
        }
    } else {
        for (int i = threadIdx.x * 4; i < k; i += 4 * THREADS) {
            const float4 v = *(const float4*)(x + i);
            *(uint32_t*)(q + (size_t)row * k + i) =
                pack4_e4m3(__fdiv_rn(v.x, s), __fdiv_rn(v.y, s), __fdiv_rn(v.z, s), __fdiv_rn(v.w, s));
        }
    }
}

// Many short rows (k <= 1024): a wave per row, four to a workgroup, no barrier and no thread without elements: 2306 x 768 4.7 -> 4.1 us, 8192 x 1024
// 11.0 -> 9.0, 8192 x 512 9.1 -> 5.5, 65536 x 128 44.9 -> 17.5; 1000 rows as fast either way, 300 x 1024 3.2 against 3.5.
__global__ void __launch_bounds__(256) quant_rowwise_wave_kernel(const float* __restrict__ src, int rows, int k, int ld, uint8_t* __restrict__ q,
                                                                 float* __restrict__ scale)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const float* x = src + (size_t)row * ld;
    float4 held[4];
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = lane * 4 + 256 * u;
        held[u] = i < k ? load_once4(x + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(held[u].x), fabsf(held[u].y)), fmaxf(fabsf(held[u].z), fabsf(held[u].w))));
    amax = wave_max(amax);
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (lane == 0) scale[row] = s;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = lane * 4 + 256 * u;
        if (i < k)
            *(uint32_t*)(q + (size_t)row * k + i) = pack4_e4m3(__fdiv_rn(held[u].x, s), __fdiv_rn(held[u].y, s), __fdiv_rn(held[u].z, s), __fdiv_rn(held[u].w, s));
    }
}

// 1 x 128 blocks: 32 lanes per (row, 128-group) (bound: HBM).  A workgroup takes one group of ROWS rows (8 or 32: a half wave
// takes every eighth row, all loads first), so that the scales, stored [k/128][rows], leave as one run of the group's row:
// taken along a row instead, every scale is a 4-byte write into a cache line of its own, which the workgroups of eight L2s
// share (few rows, whose scales lie together, are taken along the row: quant_1x128_along_rows_kernel below).  8192 x 8192: 82.3 -> 55.9 us (6.0 TB/s), 4096 x 2048: 11.3 -> 9.4.  Eight rows per workgroup where few blocks leave
// the latency of one workgroup: 512 x 4096 3.5 us against 4.0 with 32 rows, 16 x 7168 2.3 against 3.0 (4.3 along the rows);
// 2560 x 2560 8.5 against 8.3, 8192 x 8192 65 against 58.
constexpr int QUANT_1X128_FEW = 1 << 14;      // blocks up to which a workgroup takes eight rows
template <int ROWS>
__global__ void __launch_bounds__(256) quant_1x128_vec_kernel(const float* __restrict__ src, int rows, int k, int ld,
                                                              uint8_t* __restrict__ q, float* __restrict__ scale)
{
    constexpr int G = ROWS / 8;
    __shared__ float tile_scale[ROWS];
    const int groups = k >> 7, g = blockIdx.x % groups, row0 = blockIdx.x / groups * ROWS, h = threadIdx.x >> 5, l = threadIdx.x & 31;
    float4 v[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row0 + h + 8 * u < rows) v[u] = load_once4(src + (size_t)(row0 + h + 8 * u) * ld + g * 128 + 4 * l);
    }
#pragma unroll
    for (int u = 0; u < G; ++u) {
        const int row = row0 + h + 8 * u;
        float amax = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
        if (l == 0) tile_scale[h + 8 * u] = s;
        if (row < rows)
            *(uint32_t*)(q + (size_t)row * k + g * 128 + 4 * l) =
                pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
    }
    __syncthreads();
    if (threadIdx.x < ROWS && row0 + (int)threadIdx.x < rows) scale[(size_t)g * rows + row0 + threadIdx.x] = tile_scale[threadIdx.x];
}

// The same for few rows (quant_1x128_along_rows of routes.hpp): half waves take (row, group) pairs counted along the rows, so that none
// is without a row and memory is read in one run; of few rows the scales of neighbouring groups share their lines all the same.
// G pairs per half wave, all loads first: four where there are enough of them to fill the chip
// (17 x 2^20 21.0 -> 19.2 us, 65 x 2^20 71 -> 66), else one.
template <int G>
__global__ void __launch_bounds__(256) quant_1x128_along_rows_kernel(const float* __restrict__ src, int rows, int k, int ld,
                                                                     uint8_t* __restrict__ q, float* __restrict__ scale)
{
    const unsigned groups = (unsigned)(k >> 7), i0 = blockIdx.x * (8u * G) + (threadIdx.x >> 5), l = threadIdx.x & 31;
    unsigned row[G], g[G];
    float4 v[G];
#pragma unroll
    for (int u = 0; u < G; ++u) {
        row[u] = (i0 + 8 * u) / groups;
        g[u] = (i0 + 8 * u) % groups;
        v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row[u] < (unsigned)rows) v[u] = load_once4(src + (size_t)row[u] * ld + g[u] * 128 + 4 * l);
    }
#pragma unroll
    for (int u = 0; u < G; ++u) {
        float amax = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
        const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
        if (row[u] >= (unsigned)rows) continue;
        if (l == 0) scale[(size_t)g[u] * rows + row[u]] = s;
        *(uint32_t*)(q + (size_t)row[u] * k + g[u] * 128 + 4 * l) =
            pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
    }
}

// 128 x 128 blocks, one workgroup per block; the block stays in registers between the amax and the quantisation (one read
// of the input: 8192 x 8192 149 -> 55 us, 2560 x 2560 39.7 -> 8.3).  Scale stored [rows/128][k/128].
__global__ void __launch_bounds__(256) quant_128x128_vec_kernel(const float* __restrict__ src, int k, int ld, uint8_t* __restrict__ q,
                                                                float* __restrict__ scale)
{
    __shared__ float part[4];
    const int gk = blockIdx.x, gr = blockIdx.y, h = threadIdx.x >> 5, l = threadIdx.x & 31;
    const float* x = src + (size_t)(gr * 128 + h) * ld + gk * 128 + 4 * l;      // + 8 u rows
    float4 v[16];
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = load_once4(x + (size_t)(8 * u) * ld);
#pragma unroll
    for (int u = 0; u < 16; ++u) amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (threadIdx.x == 0) scale[(size_t)gr * gridDim.x + gk] = s;
    uint8_t* o = q + (size_t)(gr * 128 + h) * k + gk * 128 + 4 * l;
#pragma unroll
    for (int u = 0; u < 16; ++u)
        *(uint32_t*)(o + (size_t)(8 * u) * k) =
            pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
}

// per-tensor scale over a contiguous array (ld == k) of 16-byte units (bound: HBM, two passes), in three launches:
//  1. every workgroup writes the maximum of its share, a plain store, into the first bytes of the output array, which nothing
//     has been written to yet (thousands of atomics on the scale slot, which had to be cleared by a launch of its own before,
//     took longer than the pass over the data);
//  2. one workgroup folds these into the scale;
//  3. the quantisation, from the end of the array to its start: what the first pass read last is still in the Infinity Cache.
// 2560 x 2560: 23.6 us with atomics (four launches), 15.2 here; 8192 x 8192 115.8 -> 96.8 (98.1 with four units per
// thread in pass 3, 100.1 from start to end as well); 1 x 4096 7.4 -> 5.6.
constexpr int QUANT_TENSOR_PARTS = 1024;      // workgroups of pass 1 at most
__global__ void __launch_bounds__(256) quant_tensor_amax_vec_kernel(const float4* __restrict__ src, size_t units, float* __restrict__ parts)
{
    __shared__ float part[4];
    float amax = 0.f;
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < units; i += 4 * stride) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = i + u * stride < units ? src[i + u * stride] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
    }
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) parts[blockIdx.x] = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}
__global__ void __launch_bounds__(256) quant_tensor_fold_kernel(const float* __restrict__ parts, int n, float* __restrict__ scale)
{
    __shared__ float part[4];
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < QUANT_TENSOR_PARTS / 256; ++u) {
        const int i = threadIdx.x + 256 * u;
        if (i < n) amax = fmaxf(amax, parts[i]);
    }
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
        amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
        *scale = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;
    }
}
constexpr int QUANT_TENSOR_UNITS = 2;
__global__ void __launch_bounds__(256) quant_tensor_apply_vec_kernel(const float4* __restrict__ src, size_t units,
                                                                     uint32_t* __restrict__ q, const float* __restrict__ scale)
{
    constexpr int U = QUANT_TENSOR_UNITS;
    const float s = *scale;
    const size_t i0 = (size_t)(gridDim.x - 1 - blockIdx.x) * (256 * U) + threadIdx.x;
    float4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = i0 + 256 * u < units ? load_once4((const float*)(src + i0 + 256 * u)) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (i0 + 256 * u < units)
            q[i0 + 256 * u] = pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
}
// The same in two launches, with memory of the caller's for the maxima: pass 1 over at most QUANT_TENSOR_WS_PARTS workgroups, whose maxima (a multiple of
// four of them) every wave of pass 2 folds for itself, behind its own loads.  2560 x 2560 16.2 -> 14.7 us, 276 x 2880 6.9 -> 5.7, 163 x 1380 6.7 -> 5.2
// (a launch is 2.4); 8192 x 8192 97.5 -> 97.0.  (1024 workgroups of 256 threads in pass 1 15.0 and 5.9, four units per thread in pass 2 14.9 and 6.2.)
constexpr int QUANT_TENSOR_WS_PARTS = 512;
__global__ void __launch_bounds__(512) quant_tensor_amax_ws_kernel(const float4* __restrict__ src, size_t units, float* __restrict__ parts)
{
    __shared__ float part[8];
    float amax = 0.f;
    const size_t stride = (size_t)gridDim.x * 512;
    for (size_t i = (size_t)blockIdx.x * 512 + threadIdx.x; i < units; i += 4 * stride) {
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = i + u * stride < units ? src[i + u * stride] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
    }
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < 8; ++w) amax = fmaxf(amax, part[w]);
        parts[blockIdx.x] = amax;
    }
}
__global__ void __launch_bounds__(256) quant_tensor_apply_ws_kernel(const float4* __restrict__ src, size_t units, uint32_t* __restrict__ q,
                                                                    float* __restrict__ scale, const float* __restrict__ parts, int n)
{
    constexpr int U = QUANT_TENSOR_UNITS, P = QUANT_TENSOR_WS_PARTS / 256;
    const size_t i0 = (size_t)(gridDim.x - 1 - blockIdx.x) * (256 * U) + threadIdx.x;
    float4 m[P], v[U];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const int i = (threadIdx.x & 63) * 4 + 256 * u;
        m[u] = i < n ? *(const float4*)(parts + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = i0 + 256 * u < units ? load_once4((const float*)(src + i0 + 256 * u)) : make_float4(0.f, 0.f, 0.f, 0.f);
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < P; ++u) amax = fmaxf(amax, fmaxf(fmaxf(m[u].x, m[u].y), fmaxf(m[u].z, m[u].w)));
    amax = wave_max(amax);
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (blockIdx.x == 0 && threadIdx.x == 0) *scale = s;
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (i0 + 256 * u < units)
            q[i0 + 256 * u] = pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
}
// Up to QUANT_TENSOR_ONE units: one workgroup, one launch, the array in its registers (1 x 4096 2.7 us against 6.1 in three
// launches, 4 x 4096 4.0 against 6.2; with eight units per thread 8 x 4096 5.9 against 6.3, which one compute unit's loads bound).
constexpr int QUANT_TENSOR_ONE = 4096;
__global__ void __launch_bounds__(1024) quant_tensor_one_kernel(const float4* __restrict__ src, int units, uint32_t* __restrict__ q,
                                                                float* __restrict__ scale)
{
    __shared__ float part[16];
    constexpr int U = QUANT_TENSOR_ONE / 1024;
    float4 v[U];
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = threadIdx.x + 1024 * u;
        v[u] = i < units ? load_once4((const float*)(src + i)) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w))));
    amax = wave_max(amax);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
    __syncthreads();
    amax = part[0];
#pragma unroll
    for (int w = 1; w < 16; ++w) amax = fmaxf(amax, part[w]);
    const float s = amax > 0.f ? __fdiv_rn(amax, 448.0f) : 1.0f;   // an all-zero group keeps scale 1
    if (threadIdx.x == 0) *scale = s;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = threadIdx.x + 1024 * u;
        if (i < units) q[i] = pack4_e4m3(__fdiv_rn(v[u].x, s), __fdiv_rn(v[u].y, s), __fdiv_rn(v[u].z, s), __fdiv_rn(v[u].w, s));
    }
}

// One launch for one or two scale arrays (the A-side and the B-side scales of a GEMM).  A group of
// 64 threads handles one 1 KiB unit (64 rows x 16 K blocks): thread r copies the 16 bytes of row r
// into LDS, then thread t gathers and writes bytes 16t..16t+15 of the unit.  256 threads = 4 units.
__global__ void __launch_bounds__(256) mx_tile_scales_kernel(const uint8_t* sf0, int rows0, int stride0, uint8_t* out0,
                                                             const uint8_t* sf1, int rows1, int stride1, uint8_t* out1,
                                                             int k)
{
    __shared__ uint8_t lds[4][64 * 16];
    const int t = threadIdx.x & 63, sub = threadIdx.x >> 6;
    size_t unit = (size_t)blockIdx.x * 4 + sub;
    const size_t units0 = mx_tiled_bytes(rows0, k) >> 10;
    const uint8_t* sf = sf0;
    uint8_t* out = out0;
    int rows = rows0, stride = stride0;
    bool live = true;
    if (unit >= units0) {
        unit -= units0;
        sf = sf1;
        out = out1;
        rows = rows1;
        stride = stride1;
        live = sf1 != nullptr && unit < (mx_tiled_bytes(rows1, k) >> 10);
    }
    const int blocks = k >> 5;
    if (live) {
        // the workgroup's four units are consecutive K groups of one 64-row block: together they read 64
        // contiguous bytes of every row (the units themselves lie K group by K group in the output)
        const int nblk = (rows + 63) >> 6, kgroups = (k + 511) >> 9;
        const int kg = (int)(unit % kgroups), blk = (int)(unit / kgroups);
        unit = (size_t)kg * nblk + blk;
        const int row = blk * 64 + t;
        const uint8_t* src = sf + (size_t)row * stride + kg * 16;
        const bool vec = row < rows && kg * 16 + 16 <= blocks && (((uintptr_t)src) & 3) == 0;
        uint32_t w[4] = {0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu};
        if (vec) {
#pragma unroll
            for (int q = 0; q < 4; ++q) w[q] = ((const uint32_t*)src)[q];
        } else if (row < rows) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t v = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) v |= (uint32_t)(kg * 16 + 4 * q + e < blocks ? src[4 * q + e] : 127u) << (8 * e);
                w[q] = v;
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) ((uint32_t*)lds[sub])[t * 4 + q] = w[q];
    }
    __syncthreads();
    if (live) {
        const int pair = t >> 5, r16 = (t >> 1) & 15;
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int st = e & 1, par = (e >> 1) & 1, jp = (e >> 2) & 1, g = (t & 1) * 2 + (e >> 3);
            const int row = 32 * jp + 8 * (r16 >> 2) + 4 * par + (r16 & 3);
            w[e >> 2] |= (uint32_t)lds[sub][row * 16 + pair * 8 + st * 4 + g] << (8 * (e & 3));
        }
        *(v4i*)(out + (unit << 10) + t * 16) = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
}

// 127 everywhere (tiled layout), for producers that then write only the real (row, block) positions.
__global__ void __launch_bounds__(256) mx_tiled_fill_kernel(uint32_t* scale, size_t dwords)
{
    const size_t d = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (d < dwords) scale[d] = 0x7f7f7f7fu;
}

}  // namespace a8w8
