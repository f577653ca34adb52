// HQQ two-per-byte codes in registers: shared by the kernels of hqq.hip and hqq_tile.hip.
#pragma once
#include "common.h"

namespace ao {

typedef _Float16 hqq_f16x2_t __attribute__((ext_vector_type(2)));

// The eight codes of a dword of four byte rows or columns -> low and high nibbles as one byte each: the byte-to-float
// conversions and byte permutes below then take them in place (shifting every code down to bit 0 first cost a third of the
// kernel's instructions).  The sign bit of a signed nibble is flipped: code = byte - 8.
template <bool SIGNED>
__device__ __forceinline__ void hqq_nibbles(uint32_t w, uint32_t& lo, uint32_t& hi) {
    lo = w & 0x0f0f0f0fu;
    hi = (w >> 4) & 0x0f0f0f0fu;
    if (SIGNED) {
        lo ^= 0x08080808u;
        hi ^= 0x08080808u;
    }
}
// fp16: codes in bytes B0 of `a` and B1 of `b` -> the weight pair (q - z) * s, each operation rounded
template <bool SIGNED, int B0, int B1>
__device__ __forceinline__ uint32_t hqq_pair(uint32_t a, uint32_t b, uint32_t s2, uint32_t z2) {
    // 0x6400 | u is the fp16 value 1024 + u, exactly: one byte permute builds the pair without a conversion
    const uint32_t m = __builtin_amdgcn_perm(b, a, 0x0c000c00u | B0 | ((4u + B1) << 16)) | 0x64006400u;
    hqq_f16x2_t q, s, z;
    __builtin_memcpy(&q, &m, 4);
    __builtin_memcpy(&s, &s2, 4);
    __builtin_memcpy(&z, &z2, 4);
    const _Float16 off = SIGNED ? (_Float16)1032.0f : (_Float16)1024.0f;
    q = q - hqq_f16x2_t{off, off};                 // exact
    const hqq_f16x2_t w = (q - z) * s;             // each op rounds to fp16
    uint32_t r;
    __builtin_memcpy(&r, &w, 4);
    return r;
}

// bf16: the weights of the nibbles at bits (0, 16) or, ODD, (4, 20) of p, as fp32 products that the caller rounds to bf16.  The masked
// nibble is the fp16 subnormal q 2^-24 (q 2^-20), which a mixed fma turns into q - z with the one rounding of the subtraction;
// with a zero low operand the conversion leaves bf16(q - z) in the high half, an fp32 again.  33 instructions for 8
// weights, where a byte conversion and a subtraction for each took 39.  SIGNED: p has its sign bits flipped, code = nibble - 8.
template <bool SIGNED, bool ODD>
__device__ __forceinline__ void hqq_products(uint32_t p, float z0, float z1, float s0, float s1, float& w0, float& w1) {
    p &= ODD ? 0x00F000F0u : 0x000F000Fu;
    const float up = ODD ? 0x1p20f : 0x1p24f;
    float t0, t1;
    if (SIGNED) {   // - 8 is exact
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(t0) : "v"(p), "s"(up), "v"(-8.0f));
        asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(t1) : "v"(p), "s"(up), "v"(-8.0f));
        t0 -= z0;
        t1 -= z1;
    } else {
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[1,0,0]" : "=v"(t0) : "v"(p), "s"(up), "v"(z0));
        asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(t1) : "v"(p), "s"(up), "v"(z1));
    }
    w0 = hw_rne_bf16(t0) * s0;
    w1 = hw_rne_bf16(t1) * s1;
}
// a dword of four bytes along n.  Columns: the (low, high) pair of bytes O and O + 2, whose columns' zeros and scales are z[O], z[O + 2] ..
template <bool SIGNED, int O>
__device__ __forceinline__ void hqq_columns2(uint32_t d, const float* z, const float* s, uint32_t& c0, uint32_t& c2) {
    if (SIGNED) d ^= 0x88888888u;
    if (O) d >>= 8;
    float l0, l2, h0, h2;
    hqq_products<SIGNED, false>(d, z[O], z[O + 2], s[O], s[O + 2], l0, l2);
    hqq_products<SIGNED, true>(d, z[O], z[O + 2], s[O], s[O + 2], h0, h2);
    c0 = hw_bf16_pack(l0, h0);
    c2 = hw_bf16_pack(l2, h2);
}
template <bool SIGNED>
__device__ __forceinline__ void hqq_columns(uint32_t d, const float* z, const float* s, uint32_t& c0, uint32_t& c1, uint32_t& c2, uint32_t& c3) {
    hqq_columns2<SIGNED, 0>(d, z, s, c0, c2);
    hqq_columns2<SIGNED, 1>(d, z, s, c1, c3);
}
// .. Row: the four low or, HIGH, high nibbles as two pairs
template <bool SIGNED, bool HIGH>
__device__ __forceinline__ void hqq_row(uint32_t d, const float* z, const float* s, uint32_t& p0, uint32_t& p1) {
    if (SIGNED) d ^= 0x88888888u;
    float w0, w1, w2, w3;
    hqq_products<SIGNED, HIGH>(d, z[0], z[2], s[0], s[2], w0, w2);
    hqq_products<SIGNED, HIGH>(d >> 8, z[1], z[3], s[1], s[3], w1, w3);
    p0 = hw_bf16_pack(w0, w1);
    p1 = hw_bf16_pack(w2, w3);
}

// Transposed product, bf16: the weights of a dword of four bytes along n in a lane whose three neighbours (lanes 4 i .. 4 i + 3) hold other byte
// rows of the same group at the same n.  The zeros and scales then belong to the four values and not to the lane, and a 4x4x4 matrix
// instruction, D[i] of lane j = sum over k of A(lane i)[k] * B(lane j)[k] + C[i] within four lanes, applies them to all values at once:
//   t = q - z     B: the masked nibbles, fp16 subnormals q 2^-24 or q 2^-20, in the order of bytes 0, 2, 1, 3;  A: 2^15 or 2^11 where it puts
//                 them in order;  C = -z 2^-9, itself such a product.  One value is rounded to fp32 once, then to bf16: bf16(t) 2^-9.
//   w = t * s     A: the scales on the diagonal; the product of two bf16 is exact.  Rounded: w 2^-9.
// The caller multiplies its sums by DOWN.  13 VALU and 4 two-pass matrix instructions for 8 weights, where mixed fmas and
// multiplications take 37 VALU (32 rows x 4096 x 11008 18.2 -> 17.6 us by this alone).  For scales and zeros in HqqOrdinary's range only, whose weights (0
// or 2^-80 .. 2^81) the factor leaves exact: beyond it bf16(t * s) may overflow, which 2^-9 of it does not, or be a subnormal on the way, and the zeros off
// the diagonal meet an infinite z as 0 * inf, a NaN for its three neighbours.
typedef float hqq_f4_t __attribute__((ext_vector_type(4)));
typedef _Float16 hqq_f16x4_t __attribute__((ext_vector_type(4)));
typedef short hqq_s16x4_t __attribute__((ext_vector_type(4)));
struct HqqRowScales { hqq_s16x4_t s; hqq_f4_t z; };   // the diagonal of scales, -z 2^-9
struct HqqRowMatrices {
    static constexpr float DOWN = 512.0f;
    uint32_t m0, m1;                  // this lane's place on the diagonal
    hqq_f16x4_t low, high;            // the nibbles at bits 0 and 4
    hqq_s16x4_t zero;                 // -2^-9 on the diagonal
    static __device__ __forceinline__ uint2 pair(uint32_t a, uint32_t b) { return make_uint2(a, b); }
    __device__ __forceinline__ explicit HqqRowMatrices(int lane) {
        const int i = lane & 3;
        m0 = i == 0 ? 0xffffu : i == 1 ? 0xffff0000u : 0u;
        m1 = i == 2 ? 0xffffu : i == 3 ? 0xffff0000u : 0u;
        // lane i takes byte i, which is operand 0, 2, 1, 3
        const uint32_t n0 = i == 0 ? 0xffffu : i == 2 ? 0xffff0000u : 0u, n1 = i == 1 ? 0xffffu : i == 3 ? 0xffff0000u : 0u;
        low = __builtin_bit_cast(hqq_f16x4_t, pair(n0 & 0x78007800u, n1 & 0x78007800u));     // 2^15
        high = __builtin_bit_cast(hqq_f16x4_t, pair(n0 & 0x68006800u, n1 & 0x68006800u));    // 2^11
        zero = __builtin_bit_cast(hqq_s16x4_t, pair(m0 & 0xBB00BB00u, m1 & 0xBB00BB00u));
    }
    __device__ __forceinline__ HqqRowScales scales(uint32_t s0, uint32_t s1, uint32_t z0, uint32_t z1) const {
        return HqqRowScales{__builtin_bit_cast(hqq_s16x4_t, pair(s0 & m0, s1 & m1)),
                            __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(zero, __builtin_bit_cast(hqq_s16x4_t, pair(z0, z1)), hqq_f4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0)};
    }
    // two pairs of low and two of high nibbles' weights, 2^-9 of them
    template <bool SIGNED>
    __device__ __forceinline__ void weights(uint32_t d, const HqqRowScales& c, uint32_t& lo0, uint32_t& lo1, uint32_t& hi0, uint32_t& hi1) const {
        if (SIGNED) d ^= 0x88888888u;
        const uint32_t e = d >> 8;
        auto half = [&](uint32_t b0, uint32_t b1, hqq_f16x4_t a, uint32_t& w0, uint32_t& w1) {
            hqq_f16x4_t q = __builtin_bit_cast(hqq_f16x4_t, pair(b0, b1));
            const hqq_f4_t t = __builtin_amdgcn_mfma_f32_4x4x4f16(a, q, c.z, 0, 0, 0);
            const hqq_f4_t w = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(c.s, __builtin_bit_cast(hqq_s16x4_t, pair(hw_bf16_pack(t.x, t.y), hw_bf16_pack(t.z, t.w))),
                                                                      hqq_f4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            w0 = hw_bf16_pack(w.x, w.y);
            w1 = hw_bf16_pack(w.z, w.w);
        };
        uint32_t l0 = d & 0x000F000Fu, l1 = e & 0x000F000Fu, h0 = d & 0x00F000F0u, h1 = e & 0x00F000F0u;
        if (SIGNED) {   // the sign bit was flipped: code - 8, exact among the subnormals
            auto less = [](uint32_t p, uint32_t eight) {
                return __builtin_bit_cast(uint32_t, __builtin_bit_cast(hqq_f16x2_t, p) - __builtin_bit_cast(hqq_f16x2_t, eight));
            };
            l0 = less(l0, 0x00080008u); l1 = less(l1, 0x00080008u);
            h0 = less(h0, 0x00800080u); h1 = less(h1, 0x00800080u);
        }
        half(l0, l1, low, lo0, lo1);
        half(h0, h1, high, hi0, hi1);
    }
};

// Whether every scale and zero seen is 2^-40 .. 2^40 in magnitude, or 0, both 16 bits of a dword at once: two instructions a dword, which know no
// 0; a wave that met something else looks again.
typedef uint16_t hqq_u16x2_t __attribute__((ext_vector_type(2)));
struct HqqOrdinary {
    static constexpr uint16_t LO = (127 - 40) << 7, HI = (127 + 40) << 7;
    hqq_u16x2_t most = {0, 0};   // of twice the magnitude's bits less 2 LO, where a magnitude below LO wraps beyond all others
    __device__ __forceinline__ void see(uint32_t d) {
        const hqq_u16x2_t b = __builtin_bit_cast(hqq_u16x2_t, d) * (uint16_t)2 - hqq_u16x2_t{2 * LO, 2 * LO};
        most = __builtin_elementwise_max(most, b);
    }
    __device__ __forceinline__ bool all() const { return most.x <= 2 * (HI - LO) && most.y <= 2 * (HI - LO); }
    static __device__ __forceinline__ bool with_zeros(uint32_t d) {
        const uint32_t lo = d & 0x7fffu, hi = (d >> 16) & 0x7fffu;
        return (lo == 0 || (lo >= LO && lo <= HI)) && (hi == 0 || (hi >= LO && hi <= HI));
    }
};

// fp32 partial sums [slices][count] added and rounded to bf16 or fp16
void launch_hqq_finish(const float* part, int slices, int64_t count, bool bf16, uint16_t* y, hipStream_t st);

// hqq_tile.hip: the product on 32- to 96-row tiles.  The plan's `rows` is 0 where it does not take the problem.
struct HqqTilePlan { int rows, tiles_m, tiles_n, parts; double us; };
HqqTilePlan hqq_tile_plan(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed, bool bf16, int max_parts = 16);
HqqTilePlan hqq_tile_route(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed, bool bf16);   // .. or is not the fastest
double hqq_stream_us(int64_t M, int64_t K, int64_t N, int64_t group, bool transposed);   // the streaming kernel's estimate, of its plan's costs
void launch_hqq_tile(const HqqTilePlan& p, const uint8_t* packed, const uint16_t* scales, const uint16_t* zeros, const uint16_t* a, int64_t lda,
                     int64_t M, int64_t K, int64_t N, int64_t group, bool is_signed, bool bf16, bool transposed, float* part, uint16_t* y,
                     hipStream_t st);

}  // namespace ao
