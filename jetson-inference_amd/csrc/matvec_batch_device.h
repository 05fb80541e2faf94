// Weight decode and matrix-core helpers shared by the batched GEMVs
// (matvec_batch.hip) and the prompt matrix products (prefill.hip): block
// codes as exact fp16 fragments, in the element order that both kernels' x
// fragments use.
#pragma once

#include "jinf_device.h"
#include "quant_device.h"

namespace jinf {
namespace {

typedef _Float16 mb_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 mb_h2 __attribute__((ext_vector_type(2)));
typedef float mb_f16 __attribute__((ext_vector_type(16)));
typedef float mb_f4 __attribute__((ext_vector_type(4)));

constexpr int kMbCols = 256;      // columns per slab

// Bytes of one row's 256-column slab.
template <int QT> struct MbFmt;
template <> struct MbFmt<kQ4_0> { static constexpr int SB = 144; };
template <> struct MbFmt<kQ8_0> { static constexpr int SB = 272; };
template <> struct MbFmt<kQ4_K> { static constexpr int SB = 144; };
template <> struct MbFmt<kQ6_K> { static constexpr int SB = 210; };
// 16-byte chunks that cover one row's slab: Q4_0, Q8_0 and Q4_K slabs
// (144 / 272 / 144 bytes) start 16-byte aligned in a 16-byte aligned matrix;
// a Q6_K slab (210 bytes) starts at an even offset, so 14 chunks cover it.
template <int QT> constexpr int mb_nch() { return QT == kQ6_K ? 14 : MbFmt<QT>::SB / 16; }

// Two 16-bit LDS reads (2-byte aligned) as one word.  (One 32-bit read at
// the 2-byte aligned address gives the same word, but unaligned LDS reads
// are slower: 116 against 111 us over the four batch-32 GEMVs of a layer.)
__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) {
    const uint16_t* q = reinterpret_cast<const uint16_t*>(p);
    return (uint32_t)q[0] | ((uint32_t)q[1] << 16);
}
__device__ __forceinline__ uint32_t lds_u16(const uint8_t* p) {
    return *reinterpret_cast<const uint16_t*>(p);
}

__device__ __forceinline__ mb_h2 as_h2(uint32_t u) { return __builtin_bit_cast(mb_h2, u); }

// Eight 4-bit codes (four bytes, element 2 i in the low nibble of byte i)
// as fp16 (q + bias) in the order (0, 4, 1, 5, 2, 6, 3, 7); `hi2` adds two
// high bits per element (Q6_K: the pair masks of element i and i + 4).
__device__ __forceinline__ mb_h8 mb_nibbles(uint32_t w, uint32_t hi2, float bias) {
    const mb_h2 b = mb_h2{(_Float16)(-1024.0f + bias), (_Float16)(-1024.0f + bias)};
    mb_h2 p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // (w >> 4 i) & 0x000F000F | 0x64006400 in one instruction
        uint32_t v = __builtin_amdgcn_bitop3_b32(w >> (4 * i), 0x000F000Fu, 0x64006400u, 0xEA);
        v |= ((hi2 >> (2 * i)) & 0x00030003u) << 4;
        p[i] = as_h2(v) + b;  // (1024 + q) + (bias - 1024): exact
    }
    return mb_h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// Eight 4-bit codes q times an integer sub-block scale g <= 63 as fp16 g q,
// in the order of mb_nibbles: one packed FMA per pair, (1024 + q) g +
// (-1024 g), whose exact value g q <= 945 is representable, so its one
// rounding changes nothing.
__device__ __forceinline__ mb_h8 mb_nibbles_scaled(uint32_t w, _Float16 g) {
    const mb_h2 g2 = mb_h2{g, g};
    const mb_h2 c = mb_h2{(_Float16)-1024.0f, (_Float16)-1024.0f} * g2;  // exact: g < 64
    mb_h2 p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = __builtin_amdgcn_bitop3_b32(w >> (4 * i), 0x000F000Fu, 0x64006400u, 0xEA);
        p[i] = __builtin_elementwise_fma(as_h2(v), g2, c);
    }
    return mb_h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// Eight 4-bit codes as fp16 g (q - 8) (integer g <= 63), in the order of
// mb_nibbles: the code goes to mantissa bits 6 .. 9 of 16 + q, and one packed
// FMA gives (16 + q) g - 24 g, exact throughout (24 g <= 1512 has 8
// significant bits).
__device__ __forceinline__ mb_h8 mb_nibbles_centered(uint32_t w, _Float16 g) {
    const mb_h2 g2 = mb_h2{g, g};
    const mb_h2 c = mb_h2{(_Float16)-24.0f, (_Float16)-24.0f} * g2;
    const uint32_t sh[4] = {w << 6, w << 2, w >> 2, w >> 6};
    mb_h2 p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = __builtin_amdgcn_bitop3_b32(sh[i], 0x03C003C0u, 0x4C004C00u, 0xEA);
        p[i] = __builtin_elementwise_fma(as_h2(v), g2, c);
    }
    return mb_h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// Eight int8 codes (two words) as fp16 in the order (0, 4, 1, 5, 2, 6, 3, 7).
__device__ __forceinline__ mb_h8 mb_int8(uint32_t w0, uint32_t w1) {
    const mb_h2 b = mb_h2{(_Float16)-1152.0f, (_Float16)-1152.0f};
    mb_h2 p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // byte i of w0 -> byte 0, byte i of w1 -> byte 2, zero elsewhere
        const uint32_t sel = (uint32_t)i | 0x0C00u | ((uint32_t)(4 + i) << 16) | 0x0C000000u;
        const uint32_t v = __builtin_amdgcn_perm(w1, w0, sel);
        p[i] = as_h2((v ^ 0x00800080u) | 0x64006400u) + b;  // 1024 + (q + 128) - 1152
    }
    return mb_h8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

__device__ __forceinline__ mb_f16 mfma(mb_h8 a, mb_h8 b, mb_f16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Token of accumulator register r in lane half h of M-tile mt
// (v_mfma_f32_32x32x* D layout: row 8 (r / 4) + 4 h + r % 4).
__device__ __forceinline__ int mb_token(int mt, int r, int h) {
    return 32 * mt + 8 * (r >> 2) + 4 * h + (r & 3);
}

// RMSNorm weights of 8-column group g (1 without a norm): 16-byte loads when
// the weights are 16-byte aligned, else element loads.
__device__ __forceinline__ void mb_norm8(const void* norm_w, int norm_f16, int g, float (&gw)[8]) {
    if (!norm_w) {
#pragma unroll
        for (int e = 0; e < 8; ++e) gw[e] = 1.0f;
    } else if (((uintptr_t)norm_w & 15) != 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            gw[e] = norm_f16 ? h2f(static_cast<const uint16_t*>(norm_w)[8 * g + e])
                             : static_cast<const float*>(norm_w)[8 * g + e];
    } else if (norm_f16) {
        const uint4 q = *(static_cast<const uint4*>(norm_w) + g);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            gw[2 * i] = h2f((uint16_t)(w[i] & 0xFFFFu));
            gw[2 * i + 1] = h2f((uint16_t)(w[i] >> 16));
        }
    } else {
        const float4 p = *(static_cast<const float4*>(norm_w) + 2 * g);
        const float4 q = *(static_cast<const float4*>(norm_w) + 2 * g + 1);
        gw[0] = p.x; gw[1] = p.y; gw[2] = p.z; gw[3] = p.w;
        gw[4] = q.x; gw[5] = q.y; gw[6] = q.z; gw[7] = q.w;
    }
}

}  // namespace
}  // namespace jinf
