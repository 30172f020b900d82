// What the expert kernels of long passes share: rows of activations as matrix-core operands, a row's own bytes together.
//
// For the list kernels a row of k columns is [sub-block of 32] x 128 bytes (list_block), the eight columns of a block in slot
// order [0, 2, 1, 3, 4, 6, 5, 7] (the order a payload dword's nibbles come out of the masks), its sums over the sub-blocks
// float32, in bfloat16 parts (list_sum_put), its values scaled (binary16_parts).  moe_long.hip's rows: long_tiles.hpp.
#pragma once
#include "shv_device.hpp"

namespace shv_moe {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStSubBytes = 128;  // a row's sub-block: 2 parts x 4 column blocks x 16 bytes

__host__ __device__ constexpr size_t staged_sums_offset(int rows, int k) { return static_cast<size_t>(rows) * (k / 32) * 128; }
// Where a pair's act row comes as operands (moe_long.hip): its sub-blocks' sums, in the library's scratch.
__host__ __device__ constexpr size_t packed_sums_bytes(long long pairs, int ffn) { return static_cast<size_t>(pairs) * (ffn / 256) * 32; }

// v as the exact sum of three bfloat16 values (bit patterns): eight bits of it each, cut off, so that what is left is exact.
__device__ __forceinline__ void bf16_parts(float v, uint16_t &p0, uint16_t &p1, uint16_t &p2) {
    const uint32_t b0 = __float_as_uint(v);
    const float r1 = v - __uint_as_float(b0 & 0xFFFF0000u);
    const uint32_t b1 = __float_as_uint(r1);
    const float r2 = r1 - __uint_as_float(b1 & 0xFFFF0000u);
    p0 = static_cast<uint16_t>(b0 >> 16);
    p1 = static_cast<uint16_t>(b1 >> 16);
    p2 = static_cast<uint16_t>(__float_as_uint(r2) >> 16);
}
// The parts of two values side by side: first parts, second, third, two zeros.
__device__ __forceinline__ u32x4_t bf16_parts_pair(float a, float b) {
    uint16_t a0, a1, a2, b0, b1, b2;
    bf16_parts(a, a0, a1, a2);
    bf16_parts(b, b0, b1, b2);
    return u32x4_t{a0 | static_cast<uint32_t>(b0) << 16, a1 | static_cast<uint32_t>(b1) << 16, a2 | static_cast<uint32_t>(b2) << 16, 0u};
}
// Two whole numbers below 256 (a sub-block's min is below 64) as a pair of bfloat16 values, exact.
__device__ __forceinline__ uint32_t bf16_pair(uint32_t a, uint32_t b) {
    return (__float_as_uint(static_cast<float>(a)) >> 16) | (__float_as_uint(static_cast<float>(b)) & 0xFFFF0000u);
}

// Where the high part of columns 32 sub + 8 c .. + 7 lies in a row staged for the list kernels; its low part is 64 bytes on.
// [super-block][low / high nibbles' sub-blocks][c][part][group]: what the lanes of one operand take of a token is a line.
__host__ __device__ constexpr int list_block(int sub, int c) { return (sub >> 3) * 1024 + (sub & 1) * 512 + c * 128 + ((sub >> 1) & 3) * 16; }

// The sums of a row staged for the list kernels: [super-block] x 64 bytes, [part 0, 1][group] x 8 bytes, the group's two
// sub-blocks' first and second bfloat16 parts in part 0, their third in part 1 (and two zeros, which its owner writes).
// Then the rows' exponents, an int each; of SwiGLU rows, whose sub-blocks have one each, a byte each.
constexpr int kListSumBytes = 64;
__host__ __device__ constexpr size_t list_exps_offset(int rows, int k) { return staged_sums_offset(rows, k) + static_cast<size_t>(rows) * (k / 256) * kListSumBytes; }
__host__ __device__ constexpr size_t list_bytes(int rows, int k) { return list_exps_offset(rows, k) + static_cast<size_t>(rows) * sizeof(int32_t); }
__host__ __device__ constexpr size_t list_act_exps_offset(long long pairs, int ffn) { return static_cast<size_t>(pairs) * (ffn / 256) * kListSumBytes; }
__host__ __device__ constexpr size_t list_act_bytes(long long pairs, int ffn) { return list_act_exps_offset(pairs, ffn) + static_cast<size_t>(pairs) * (ffn / 32); }
__device__ __forceinline__ void list_sum_put(char *sb_sums, int sub, float sum) {
    uint16_t *p = reinterpret_cast<uint16_t *>(sb_sums + ((sub >> 1) & 3) * 8) + (sub & 1);
    bf16_parts(sum, p[0], p[2], p[16]);
    p[18] = 0;
}

// The list kernels' values: times the power of two 2^(kListOne - e) that brings the largest of their row (of their sub-block)
// to 2^14 .. 2^15, e being its biased exponent, as two binary16 parts: 22 bits or more of anything down to 2^-17 of the largest,
// whatever their size (unscaled, values of 1e-4 keep 11 to 12 bits and values past 65504 none).
constexpr int kListOne = 127 + 14;
__device__ __forceinline__ int biased_exponent(float largest) { return __float_as_uint(largest) >> 23 & 255; }
__device__ __forceinline__ void binary16_parts(float u, _Float16 &hi, _Float16 &lo) {
    hi = static_cast<_Float16>(u);
    lo = fabsf(u) < INFINITY ? static_cast<_Float16>(u - static_cast<float>(hi)) : static_cast<_Float16>(0.f);  // an infinity is all in hi
}

// Four columns c .. c + 3 of row t for the list kernels, e the row's exponent, and (the lane of the first of 64)
// the sums of two sub-blocks; the sixteen lanes of the two are neighbours and all here.
__device__ __forceinline__ void stage_list_quad(const float4 v, int e, int t, int c, int k, int rows, char *staged) {
    const float o[4] = {ldexpf(v.x, kListOne - e), ldexpf(v.z, kListOne - e), ldexpf(v.y, kListOne - e), ldexpf(v.w, kListOne - e)};
    half4_t h, l;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        _Float16 hi, lo;
        binary16_parts(o[j], hi, lo);
        h[j] = hi;
        l[j] = lo;
    }
    char *at = staged + static_cast<size_t>(t) * (k / 32) * kStSubBytes + list_block(c >> 5, (c & 31) >> 3) + ((c & 7) >> 2) * 8;
    *reinterpret_cast<half4_t *>(at) = h;
    *reinterpret_cast<half4_t *>(at + 64) = l;
    const float sum = shv::sum8_all((o[0] + o[2]) + (o[1] + o[3]));
    const u32x4_t p = bf16_parts_pair(sum, shv::dpp_f32<shv::kDppMirror>(sum));  // and of the sub-block after it, which the next eight lanes hold
    if ((c & 63) == 0) {
        char *sums = staged + staged_sums_offset(rows, k) + (static_cast<size_t>(t) * (k / 256) + (c >> 8)) * kListSumBytes + ((c >> 6) & 3) * 8;
        *reinterpret_cast<u32x2_t *>(sums) = u32x2_t{p.x, p.y};
        *reinterpret_cast<u32x2_t *>(sums + 32) = u32x2_t{p.z, p.w};
    }
}

// The masks and exponents of the two nibble positions a weight is read from.
struct NibbleMasks {
    uint32_t m0, m4;  // bits 0..3, 4..7 of both halves
    uint32_t o0, o4;  // the halves 1024, 64
};
__device__ __forceinline__ NibbleMasks nibble_masks() {
    NibbleMasks c;
    c.m0 = 0x000F000Fu, c.m4 = 0x00F000F0u;
    c.o0 = 0x64006400u, c.o4 = 0x54005400u;
    // opaque to the optimiser: a mask in a scalar register and an exponent in a vector one make (q & m) | o one instruction
    asm volatile("" : "+s"(c.m0), "+s"(c.m4));
    asm volatile("" : "+v"(c.o0), "+v"(c.o4));
    return c;
}

// Eight weights of two payload dwords as n * sc: HI false the low nibbles, true the high ones.  A nibble in the low bits
// of a half's mantissa reads, under the right exponent, as C + n: bits 0..3 under 1024's, bits 4..7 under 64's (the odd
// bytes' nibbles take one shift down there).  One fused multiply-add then makes (C + n) * sc - C * sc = n * sc: a whole
// number up to 15 * 63, exact in binary16, as are C * sc.
template <bool HI>
__device__ __forceinline__ half8_t weights8(uint32_t q0, uint32_t q1, uint32_t sc, const NibbleMasks &nc) {
    const _Float16 s1 = static_cast<_Float16>(static_cast<float>(sc));
    const half2_t s2 = {s1, s1};
    half2_t w[4], c[4];
    if constexpr (!HI) {
        w[0] = __builtin_bit_cast(half2_t, (q0 & nc.m0) | nc.o0); w[1] = __builtin_bit_cast(half2_t, ((q0 >> 4) & nc.m4) | nc.o4);
        w[2] = __builtin_bit_cast(half2_t, (q1 & nc.m0) | nc.o0); w[3] = __builtin_bit_cast(half2_t, ((q1 >> 4) & nc.m4) | nc.o4);
        c[0] = c[2] = s2 * static_cast<half2_t>(static_cast<_Float16>(-1024.f));
        c[1] = c[3] = s2 * static_cast<half2_t>(static_cast<_Float16>(-64.f));
    } else {
        w[0] = __builtin_bit_cast(half2_t, (q0 & nc.m4) | nc.o4); w[1] = __builtin_bit_cast(half2_t, ((q0 >> 8) & nc.m4) | nc.o4);
        w[2] = __builtin_bit_cast(half2_t, (q1 & nc.m4) | nc.o4); w[3] = __builtin_bit_cast(half2_t, ((q1 >> 8) & nc.m4) | nc.o4);
        c[0] = c[1] = c[2] = c[3] = s2 * static_cast<half2_t>(static_cast<_Float16>(-64.f));
    }
    half8_t b;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const half2_t p = __builtin_elementwise_fma(w[i], s2, c[i]);
        b[2 * i] = p[0];
        b[2 * i + 1] = p[1];
    }
    return b;
}

}  // namespace shv_moe
