// Prompt matrix products: a layer's projections over up to kPfMaxRows tokens
// of one prompt (the reference runs them one token at a time,
// src/engine.cpp:429-508).
//
//   y[t, r] = sum_c W[r, c] x[t, c]      W in Q4_0 / Q8_0 / Q4_K / Q6_K blocks
//
// Arithmetic: that of the batched GEMVs (matvec_batch.hip).  The weights'
// integer codes are exact in fp16, x is split into fp16 hi + lo under a
// power-of-two scale per token and 256-column slab (about 22 significant bits
// of every element down to 2^-18 of its slab's largest), the products run on
// v_mfma_f32_32x32x16_f16 and block scales multiply the fp32 block sums.
//
// What bounds it: with hundreds of tokens the matrix cores and the vector
// ALUs' issue.  One 32-column block of a 32 x 32 tile is 4 matrix-core
// instructions (hi and lo of two 16-column steps, 32 cycles each) and 16
// block-scale FMAs; a matrix-core instruction leaves room for about 4.5
// vector instructions beside it (measured from registers: 16 of them alone
// 526 cycles, with 64 FMAs 552, 128 646, 192 833; v_fma_mix_f32 and packed
// fp16 at half rate), so the loop's other vector work, the decode of each
// weight code, has to be spread over as many tokens as possible.  Hence the
// tile: a workgroup takes 128 tokens x 256 weight rows and decodes each
// weight once, into fragments in LDS that the two token halves' waves share;
// a wave takes 64 tokens x 64 rows (2 x 2 tiles of 32 x 32).  1000 tokens
// (Q4_0): 4096 x 14336 235 us, 28672 x 4096 565 us, 485 on a faster card (1.0
// and 0.83 PFLOP/s of matrix-core work; a dense 8192-cube fp16 library product reaches 1.2 on the
// same card, and all-zero operands run 20% faster, so part of the distance to
// the 2.4 of the probe is the clock under load); as 16 batched steps of 64
// tokens the same products take 296 and 860 us.
//
// Sums: MFMA chains of one block (hi products first: the lo ones added first
// measured a 35% larger error), scaled into a first-level sum of a slab, those
// times the slab's 1 / s into a second; except in gate / up, and in residual
// adds of Q6_K, what the second level's additions round away is carried along
// (Q6_K there sums half slabs, as it has twice the blocks).  Error against
// fp64 relative to that of batched steps (a layer's logits, fp32 cache, 72, 300
// and 1000 tokens, 1024 to 4096 columns): Q4_0 and Q8_0 0.92-1.00, Q4_K
// 0.45-0.54, Q6_K 0.87-1.01; 1000 tokens of 4096 / 14336 with an fp16 cache
// 0.88-0.96 (Q4_K 0.59).  Tried: first-level sums of two slabs under one scale
// per row, 3 to 4% faster at 1000 tokens (Q6_K 6%), but up to 1.07, and small
// columns of the output and down projections' inputs beside ones 2^22 times
// larger three to four times the error, as the batched steps scale each column
// split by itself; without the carry, 2 to 2.5% faster, but 1.01 and with the
// fp16 cache 1.04-1.16 at 1000 tokens of 4096 / 14336.
// Q4_K's minimum goes in through its codes' centre: coefficient and 32-column
// sums of x as fp16 hi + lo (the batched steps': fp32), which the centred
// codes' smaller terms more than make up for (medians with every minimum
// zeroed, where centring gains nothing: 0.97-1.07).
//
// Data movement per stage (64 columns): x fragments (hi and lo) go to LDS
// with direct-to-LDS loads; each lane loads one 32-column block of one weight
// row into registers, decodes it a stage later into LDS; both double-buffered,
// one barrier per stage.  Raw weight bytes staged in LDS and decoded by each
// wave for itself: 625 against 590 us (28672 x 4096, four whole rounds).
//
// Workgroup order: consecutive workgroups go to different XCDs, each with its
// own L2, so each XCD takes a contiguous range of (row tile, token tile)
// items with the token tile fastest: the 32 workgroups it runs together share
// a few row tiles' weights and the token tiles' x slabs.
#include <hip/hip_runtime.h>
#include <math.h>

#include "jinf_device.h"
#include "jinf_host.h"
#include "jinf/kernels_ext.h"
#include "matvec_batch_device.h"
#include "matvec_batch_internal.h"
#include "prefill_internal.h"
#include "rope_device.h"

namespace jinf {
namespace {

// One record per (32-token tile, 256-column slab): [16 k-steps][hi, lo][64
// lanes] 16-byte fragments as in the batched GEMVs' records, then (Q4_K) one
// fragment of the sub-block sums: lane t holds token t's 8 sums' hi halves,
// lane 32 + t their lo halves, scaled by 2^-5 (a sum of 32 scaled values is
// below 2^20).
constexpr int kPfRec = 33 * 1024;
constexpr float kPfSumScale = 0.03125f;
constexpr int kPfTarget = 256;  // workgroups (one per CU) that column splits aim for

enum PfEpi { kPfAdd = 0, kPfSwiGLU = 1, kPfQKV = 2 };

struct PfJob {
    int rows;              // virtual rows (kPfSwiGLU: output rows)
    int n_slabs, slabs_per_split, k_splits;
    int n_nt, n_mt;
    int full_per_xcd, tail0, tail_items, tail_per_xcd;
    int T;
    const uint8_t* W[3];
    int seg_end[3];
    int accum;
    int64_t row_bytes;
    const uint8_t* rec;
    const float* xs;
    float* y;
    int ld_y;
    float* part;           // partial sums of split tiles: [k_splits][T][rows] when
    int pend;              // left pending, else [tile - tail0][k_splits][128][256]
    // kPfQKV
    const float2* cs;
    const int32_t* pos;
    void* kc;
    void* vc;
    int kv_f16, kv_dim, head_dim, max_ctx;
};

// ---- x preparation ----

// Merges k pending partial sums into 8 columns of a row, in split order.
__device__ __forceinline__ void pf_add_parts(float (&v)[8], const float* __restrict__ pp, int k,
                                             int64_t stride) {
    float sum[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int s = 0; s < k; ++s) {
        const float4 a = *reinterpret_cast<const float4*>(pp + s * stride);
        const float4 b = *reinterpret_cast<const float4*>(pp + s * stride + 4);
        sum[0] += a.x; sum[1] += a.y; sum[2] += a.z; sum[3] += a.w;
        sum[4] += b.x; sum[5] += b.y; sum[6] += b.z; sum[7] += b.w;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += sum[e];
}

__device__ __forceinline__ void pf_load8(float (&v)[8], const float* p) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void pf_store8(float* p, const float (&v)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}

// The pending merge alone: grid (ceil(cols / 2048), T).
__global__ __launch_bounds__(256) void pf_merge_kernel(float* __restrict__ x, int ld_x, int cols,
                                                       const float* __restrict__ part, int k,
                                                       int64_t stride) {
    const int t = blockIdx.y, g = blockIdx.x * 256 + threadIdx.x;
    if (g >= cols / 8) return;
    float* xr = x + (int64_t)t * ld_x + 8 * g;
    float v[8];
    pf_load8(v, xr);
    pf_add_parts(v, part + (int64_t)t * cols + 8 * g, k, stride);
    pf_store8(xr, v);
}

// One prompt token's whole preparation in one pass: the pending merge, the
// row's RMSNorm factor (norm_w), per 256-column slab the power-of-two scale
// that puts the slab's largest prepared magnitude in [2^14, 2^15), then the
// row's share of the records, from the row held in registers (NG groups of
// 8 columns a thread).  What bounds it: with few tokens the chain load -
// reduce - store and the launch, with many the bytes.  One launch for
// statistics and one for the conversion (which read the row again) made the
// 77-token prompt of 4 layers of 2048 / 8192 791 us, this one 719; 1000
// tokens of 4096 / 14336 take the same either way (8.70 ms for 8 layers).  With
// a scale per slab, half a wave's maximum, a row without a norm needs no
// barrier: 28.5 -> 27.6 us for 1000 tokens of 14336 columns, 17.7 -> 16.8 of
// 4096 (with a norm).  A
// token owns 16 bytes of each 512-byte run of a record, so the 8 tokens of a
// 128-byte line go to workgroups of one XCD, whose L2 joins them.  Tokens
// past T, up to the next whole tile, are zeros.
template <int NG>
__global__ __launch_bounds__(256) void pf_prepare_kernel(float* __restrict__ x, int ld_x, int cols,
                                                         int T, const float* __restrict__ part,
                                                         int k, int64_t stride,
                                                         const void* __restrict__ norm_w,
                                                         int norm_f16, float eps,
                                                         float* __restrict__ xs,
                                                         uint8_t* __restrict__ rec) {
    __shared__ double red[4];
    const int xcd = blockIdx.x & 7, ix = blockIdx.x >> 3;
    const int t = 8 * (8 * (ix >> 3) + xcd) + (ix & 7), tid = threadIdx.x;
    const int ng = cols / 8;
    const bool live = t < T;
    float v[NG][8];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int g = tid + 256 * i;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = 0.0f;
        if (live && g < ng) pf_load8(v[i], x + (int64_t)t * ld_x + 8 * g);
    }
    float rs = 1.0f;
    if (live) {
        if (k > 0) {
#pragma unroll
            for (int i = 0; i < NG; ++i) {
                const int g = tid + 256 * i;
                if (g >= ng) break;
                pf_add_parts(v[i], part + (int64_t)t * cols + 8 * g, k, stride);
                pf_store8(x + (int64_t)t * ld_x + 8 * g, v[i]);
            }
        }
        if (norm_w) {
            double ss = 0.0;  // (groups past the row hold zeros)
#pragma unroll
            for (int i = 0; i < NG; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) ss = fma((double)v[i][e], (double)v[i][e], ss);
            ss = wave_sum_f64(ss);
            if ((tid & (kWave - 1)) == 0) red[tid / kWave] = ss;
            __syncthreads();
            rs = rms_scale(((red[0] + red[1]) + red[2]) + red[3], cols, eps);
        }
    }
    // group g: slab g / 32, k-step (g % 32) / 2, half g & 1
    uint8_t* rt = rec + (int64_t)(t >> 5) * (ng / 32) * kPfRec + 16 * (t & 31);
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int g = tid + 256 * i;
        if (g >= ng) break;
        if (norm_w) {
#pragma clang fp contract(off)
            float gw[8];
            mb_norm8(norm_w, norm_f16, g, gw);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = (v[i][e] * rs) * gw[e];
        }
        // the slab's scale: its 32 groups are the lanes of half a wave
        float m = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(v[i][e]));
        m = fmaxf(m, dpp_f32<0xB1>(m));
        m = fmaxf(m, dpp_f32<0x4E>(m));
        m = fmaxf(m, __shfl_xor(m, 4, kWave));
        m = fmaxf(m, dpp_f32<0x128>(m));  // row_ror:8
        m = fmaxf(m, __shfl_xor(m, 16, kWave));
        const int ex = mb_scale_exp(m);
        const float sc = ldexpf(1.0f, 15 - ex);
        if ((g & 31) == 0) {
            // (s above 2^30 is written as 0: it only scales a carried rounding
            // error, which that slab then goes without, into acc's units, and
            // has to stay in range)
            float* p = xs + ((int64_t)(t / kPfTile) * (ng / 32) + (g >> 5)) * (2 * kPfTile) + t % kPfTile;
            p[0] = ldexpf(1.0f, ex - 15);
            p[kPfTile] = sc <= 0x1p30f ? sc : 0.0f;
        }
        // columns in the order (0, 4, 1, 5, 2, 6, 3, 7); the sums are of the
        // split values
        uint32_t hw[4], lw[4];
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a0 = v[i][e] * sc, a1 = v[i][4 + e] * sc;
            const _Float16 h0 = (_Float16)a0, h1 = (_Float16)a1;
            const _Float16 l0 = (_Float16)(a0 - (float)h0), l1 = (_Float16)(a1 - (float)h1);
            hw[e] = (uint32_t)__builtin_bit_cast(uint16_t, h0) |
                    ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
            lw[e] = (uint32_t)__builtin_bit_cast(uint16_t, l0) |
                    ((uint32_t)__builtin_bit_cast(uint16_t, l1) << 16);
            sum += ((float)h0 + (float)l0) + ((float)h1 + (float)l1);
        }
        uint8_t* r = rt + (int64_t)(g >> 5) * kPfRec;
        uint8_t* fr = r + 1024 * (g & 30) + 512 * (g & 1);
        *reinterpret_cast<uint4*>(fr) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
        *reinterpret_cast<uint4*>(fr + 1024) = make_uint4(lw[0], lw[1], lw[2], lw[3]);
        // a 32-column sub-block is 4 consecutive lanes' groups
        sum += dpp_f32<0xB1>(sum);  // the halves of a k-step
        sum += dpp_f32<0x4E>(sum);  // its two k-steps
        if ((g & 3) < 2) {
            const float s = sum * kPfSumScale;
            const _Float16 hi = (_Float16)s;
            const _Float16 o = (g & 3) == 0 ? hi : (_Float16)(s - (float)hi);
            *reinterpret_cast<_Float16*>(r + 32768 + 512 * (g & 1) + 2 * ((g & 31) >> 2)) = o;
        }
    }
}

__global__ __launch_bounds__(256) void pf_rope_table_kernel(float2* __restrict__ cs,
                                                            const int32_t* __restrict__ pos,
                                                            int n, int half, RopeTheta th) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    cs[i] = rope_cs(pos[i / half], th.t[i % half]);
}

// ---- the matrix product ----

// One 16-byte direct-to-LDS load per lane from a wave-uniform base plus a
// 32-bit lane offset (see lds_load16).
__device__ __forceinline__ void pf_lds_load(const uint8_t* base, uint32_t voff,
                                            const void* lds_base) {
    const uint32_t off = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds_base;
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %3\n\t"
        "global_load_lds_dwordx4 %1, %2\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(voff), "s"(base), "s"(__builtin_amdgcn_readfirstlane(off))
        : "memory");
}

// Row lr of row tile nt: lr = 64 n + 32 i + c is wave column n's tile i, lane
// c.  kPfSwiGLU: tile 0 gate rows, tile 1 the same rows of up.
template <int EPI, int NW>
__device__ __forceinline__ const uint8_t* pf_row(const PfJob& j, int nt, int lr) {
    if constexpr (EPI == kPfSwiGLU) {
        int r = nt * 32 * NW + (lr >> 6) * 32 + (lr & 31);
        r = r < j.rows ? r : j.rows - 1;
        return ((lr >> 5) & 1 ? j.W[1] : j.W[0]) + (int64_t)r * j.row_bytes;
    } else {
        int v = nt * 64 * NW + lr;
        v = v < j.rows ? v : j.rows - 1;
        const uint8_t* base = v < j.seg_end[0] ? j.W[0] : v < j.seg_end[1] ? j.W[1] : j.W[2];
        const int start = v < j.seg_end[0] ? 0 : v < j.seg_end[1] ? j.seg_end[0] : j.seg_end[1];
        return base + (int64_t)(v - start) * j.row_bytes;
    }
}

// Segment of virtual row `row` and the row inside its own matrix.
__device__ __forceinline__ int pf_segment(int row, int e0, int e1, int* local) {
    *local = row < e0 ? row : row < e1 ? row - e0 : row - e1;
    return row < e0 ? 0 : row < e1 ? 1 : 2;
}

// A lane's share of a stage's weights: one row's 32-column block.
template <int QT> struct PfRaw;
template <> struct PfRaw<kQ4_0> { uint4 q; uint16_t d; };
template <> struct PfRaw<kQ8_0> { uint4 q[2]; uint16_t d; };
template <> struct PfRaw<kQ4_K> { uint4 q, head; };
template <> struct PfRaw<kQ6_K> { uint4 ql; uint2 qh; uint16_t sc, d; };

template <typename T>
__device__ __forceinline__ T pf_load(const uint8_t* p) {
    T v;
    __builtin_memcpy(&v, p, sizeof(T));  // any alignment
    return v;
}

// Block b (32 columns) of the row at p.
template <int QT>
__device__ __forceinline__ PfRaw<QT> pf_load_raw(const uint8_t* p, int b) {
    PfRaw<QT> r;
    if constexpr (QT == kQ4_0) {
        p += 18 * (int64_t)b;
        r.d = pf_load<uint16_t>(p);
        r.q = pf_load<uint4>(p + 2);
    } else if constexpr (QT == kQ8_0) {
        p += 34 * (int64_t)b;
        r.d = pf_load<uint16_t>(p);
        r.q[0] = pf_load<uint4>(p + 2);
        r.q[1] = pf_load<uint4>(p + 18);
    } else if constexpr (QT == kQ4_K) {
        p += 144 * (int64_t)(b >> 3);
        r.head = *reinterpret_cast<const uint4*>(p);
        r.q = *reinterpret_cast<const uint4*>(p + 16 + 16 * (b & 7));
    } else {
        p += 210 * (int64_t)(b >> 3);
        r.ql = pf_load<uint4>(p + 16 * (b & 7));
        r.qh = pf_load<uint2>(p + 128 + 8 * (b & 7));
        r.sc = pf_load<uint16_t>(p + 192 + 2 * (b & 7));
        r.d = pf_load<uint16_t>(p + 208);
    }
    return r;
}

// 8-column group o (0 .. 3) of a block as an exact fp16 fragment piece.
template <int QT>
__device__ __forceinline__ mb_h8 pf_decode8(const PfRaw<QT>& r, int o, _Float16 g) {
    if constexpr (QT == kQ4_0) {
        const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        return mb_nibbles(w[o], 0u, -8.0f);
    } else if constexpr (QT == kQ8_0) {
        const uint4 q = r.q[o >> 1];
        return (o & 1) ? mb_int8(q.z, q.w) : mb_int8(q.x, q.y);
    } else if constexpr (QT == kQ4_K) {
        const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
        return mb_nibbles_centered(w[o], g);
    } else {
        const uint32_t w[4] = {r.ql.x, r.ql.y, r.ql.z, r.ql.w};
        const uint32_t hq = ((o & 2) ? r.qh.y : r.qh.x) >> (16 * (o & 1));
        return mb_nibbles(w[o], (hq & 0xFFu) | ((hq & 0xFF00u) << 8), -32.0f);
    }
}

// The workgroup's shape and LDS: x and weight fragments of a stage (KST
// 16-column steps) and the blocks' scales, all double-buffered; for Q4_K also
// each slab's coefficient fragments and x sums.
template <int QT>
struct PfShape {
    static constexpr int MT = 2, NW = 4, MW = 2;  // token tiles per wave; waves along rows, tokens
    static constexpr int TILES = MT * MW;
    static constexpr int KST = 4;
    static constexpr int NSC = QT == kQ6_K ? 4 : 2;    // scales per row and stage
    static constexpr int XB = TILES * KST * 2048;
    static constexpr int WB = 2 * NW * KST * 1024;
    static constexpr int DB = NSC * 64 * NW * 4;
    static constexpr int CB = QT == kQ4_K ? 64 * NW * 36 : 0;  // hi and lo coefficients, factor
    static constexpr int SB = QT == kQ4_K ? TILES * 1024 : 0;
    static constexpr int IB = 2 * kPfTile * 4;  // a slab's 1 / s and s of the tokens
    static constexpr int LDS = 2 * (XB + WB + DB + CB + SB + IB);
    static_assert(32 * TILES == kPfTile && LDS <= 160 * 1024, "shape");
};

template <int QT, int EPI>
__global__ __launch_bounds__(512, 2) void pf_matmul_kernel(PfJob j) {
    using S = PfShape<QT>;
    constexpr int MT = S::MT, NW = S::NW, KST = S::KST, TILES = S::TILES;
    constexpr int NK = QT == kQ6_K ? 1 : 2;     // k-steps under one block scale
    constexpr int NBK = KST / NK;               // scale blocks per stage
    constexpr int NXI = TILES * KST * 2;        // x load instructions per stage
    static_assert(NXI % 8 == 0 && 2 * 64 * NW == 512, "one block of one row per lane and stage");
    extern __shared__ __attribute__((aligned(16))) uint8_t pf_lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, h = lane >> 5, col = lane & 31;
    const int n = wave % NW, mw = wave / NW;

    // Item order: XCD blockIdx % 8 takes a contiguous range of whole tiles
    // (token tile fastest), then its share of the tail's split tiles.
    const int li = blockIdx.x >> 3, xcd = blockIdx.x & 7;
    int tile, split = 0;
    if (li < j.full_per_xcd) {
        tile = xcd * j.full_per_xcd + li;
    } else {
        const int ti = xcd * j.tail_per_xcd + li - j.full_per_xcd;
        if (li - j.full_per_xcd >= j.tail_per_xcd || ti >= j.tail_items) return;
        tile = j.tail0 + ti / j.k_splits;
        split = ti % j.k_splits;
    }
    const bool whole = tile < j.tail0 || j.k_splits == 1;
    const int mtile = tile % j.n_mt, nt_ = tile / j.n_mt;
    const int s0 = whole ? 0 : split * j.slabs_per_split;
    const int s1 = whole ? j.n_slabs : min(j.n_slabs, s0 + j.slabs_per_split);

    const int st0 = 4 * s0, st1 = 4 * s1;  // stages

    uint8_t* const xbuf = pf_lds;
    uint8_t* const wbuf = xbuf + 2 * S::XB;
    uint8_t* const dbuf = wbuf + 2 * S::WB;
    uint8_t* const cbuf = dbuf + 2 * S::DB;
    uint8_t* const sbuf = cbuf + 2 * S::CB;
    uint8_t* const ibuf = sbuf + 2 * S::SB;

    // ---- weights: lane (row, block of the stage) loads 32 columns' bytes,
    // one stage ahead of decoding them into fragments, which is one stage
    // ahead of their use ----
    const int wlr = 32 * wave + (lane & 31);  // the lane's row of the tile
    const int wblk = lane >> 5;               // and its block of the stage
    const uint8_t* const wrow = pf_row<EPI, NW>(j, nt_, wlr);
    // fragments: [row tile][k-step][lane] 16 bytes; row tile = wlr / 32 = wave
    uint8_t* const wdst = wbuf + (wave * KST + 2 * wblk) * 1024 + (wlr & 31) * 16;
    PfRaw<QT> raw;
    _Float16 wg = 0;  // Q4_K: the block's 6-bit scale
    // piece o of the lane's block into buffer b; piece 0 also the scales
    auto decode = [&](int o, int b, int st) {
        if (o == 0) {
            float* dp = reinterpret_cast<float*>(dbuf + b * S::DB);
            if constexpr (QT == kQ4_0 || QT == kQ8_0) {
                dp[wblk * 64 * NW + wlr] = h2f(raw.d);
            } else if constexpr (QT == kQ6_K) {
                const float d = h2f(raw.d);
                dp[(2 * wblk) * 64 * NW + wlr] = d * (float)(int8_t)(raw.sc & 0xFFu);
                dp[(2 * wblk + 1) * 64 * NW + wlr] = d * (float)(int8_t)(raw.sc >> 8);
            } else {
                // The block is d sc (q - 8) + c with c = 8 d sc - dmin m: the
                // first part goes through the product with integer codes sc
                // (q - 8) (centred, so the two parts do not cancel), the
                // second times the block's sum of x once per slab.  c is
                // scaled by a power of two that fits the slab's coefficients
                // and split into fp16 hi + lo.
                const uint32_t hd = raw.head.x;
                const float d = h2f((uint16_t)(hd & 0xFFFFu)), dm = h2f((uint16_t)(hd >> 16));
                dp[wblk * 64 * NW + wlr] = d;
                const int sb = (2 * st + wblk) & 7;
                const uint32_t s3[3] = {raw.head.y, raw.head.z, raw.head.w};
                int sc, mn;
                {
                    // q4_K_scale_min's packing, at a lane-half-uniform index
                    const int sh = 8 * (sb & 3);
                    const uint32_t ba = s3[0] >> sh, bm = s3[1] >> sh, bc = s3[2] >> sh;
                    sc = sb < 4 ? ba & 0x3Fu : ((bc & 0x0Fu) << 2) | ((ba >> 6) & 3u);
                    mn = sb < 4 ? bm & 0x3Fu : (((bc >> 4) & 0x0Fu) << 2) | ((bm >> 6) & 3u);
                }
                wg = (_Float16)(float)sc;
                // |c| <= 63 (8 |d| + |dmin|) < 2^(ex + 6)
                int ex;
                (void)frexpf(fabsf(8.0f * d) + fabsf(dm), &ex);
                const float c = fmaf(8.0f * d, (float)sc, -(dm * (float)mn)) * ldexpf(1.0f, 6 - ex);
                const _Float16 hi = (_Float16)c, lo = (_Float16)(c - (float)hi);
                uint8_t* cp = cbuf + ((st >> 2) & 1) * S::CB;
                reinterpret_cast<_Float16*>(cp + wlr * 16)[sb] = hi;
                reinterpret_cast<_Float16*>(cp + 64 * NW * 16 + wlr * 16)[sb] = lo;
                reinterpret_cast<float*>(cp + 64 * NW * 32)[wlr] =
                    ldexpf(1.0f / kPfSumScale, ex - 6);
            }
        }
        *reinterpret_cast<mb_h8*>(wdst + b * S::WB + (o >> 1) * 1024 + (o & 1) * 512) =
            pf_decode8<QT>(raw, o, wg);
    };
    // x fragments of stage st, the scales of the first and, a stage before
    // each slab's end, of the next slab, and (Q4_K) the slab's sums in its first
    auto issue_x = [&](int st) {
        const int slab = st >> 2;
        uint8_t* dst = xbuf + (st & 1) * S::XB;
#pragma unroll
        for (int k = 0; k < NXI / 8; ++k) {
            const int a = wave + 8 * k;
            const int mt = a / (2 * KST), r = a % (2 * KST);
            pf_lds_load(j.rec + ((int64_t)(mtile * TILES + mt) * j.n_slabs + slab) * kPfRec +
                            (2 * KST * (st & 3) + r) * 1024,
                        16u * lane, dst + a * 1024);
        }
        if (wave == 7 && (st == st0 || ((st & 3) == 3 && st + 1 < st1))) {
            const int sl = st == st0 ? slab : slab + 1;
            pf_lds_load(reinterpret_cast<const uint8_t*>(j.xs + ((int64_t)mtile * j.n_slabs + sl) *
                                                                    (2 * kPfTile)),
                        16u * lane, ibuf + (sl & 1) * S::IB);
        }
        if constexpr (QT == kQ4_K) {
            if ((st & 3) == 0 && wave < TILES)
                pf_lds_load(j.rec + ((int64_t)(mtile * TILES + wave) * j.n_slabs + slab) * kPfRec + 32768,
                            16u * lane, sbuf + (slab & 1) * S::SB + wave * 1024);
        }
    };

    // Two-level sums: acc takes the blocks of kFlush stages, in units of x s,
    // then is scaled by the slab's 1 / s, added to sum and cleared.  kCarry:
    // what that addition rounds away starts the next acc instead, in its slab's
    // units.  So a value is rounded by at most 8 (Q4_0, Q8_0; Q6_K without a
    // carry, in 16-column blocks), 9 (Q4_K) or 16 (Q6_K) block FMAs of a
    // first-level sum, and then once, or without a carry by the row's 1 (Q6_K
    // 2) additions per slab, besides the matrix-core chains' own roundings.  (A
    // sum beyond fp32's range ends as NaN with a carry, as infinity without.)
    // The carry costs 4 instructions a value and slab instead of 2; gate / up,
    // 43% of the time, goes without: its second level has 16 additions at 4096
    // columns where the batched steps chain 32 blocks.
    constexpr bool kCarry = EPI == kPfQKV || (EPI == kPfAdd && QT != kQ6_K);
    constexpr int kFlush = QT == kQ6_K && !kCarry ? 2 : 4;
    mb_f16 acc[2][MT], sum[2][MT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[i][mt] = sum[i][mt] = mb_f16{};
    auto flush = [&](int slab) {
        const float* iv = reinterpret_cast<const float*>(ibuf + (slab & 1) * S::IB) +
                          32 * mw * MT + 4 * h;
        const float* nx = reinterpret_cast<const float*>(ibuf + ((slab & 1) ^ 1) * S::IB) +
                          kPfTile + 32 * mw * MT + 4 * h;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 w = *reinterpret_cast<const float4*>(iv + 32 * mt + 8 * q);
                const float f[4] = {w.x, w.y, w.z, w.w};
                float g[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (kCarry) {
                    const float4 u = *reinterpret_cast<const float4*>(nx + 32 * mt + 8 * q);
                    g[0] = u.x; g[1] = u.y; g[2] = u.z; g[3] = u.w;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = acc[i][mt][4 * q + e], old = sum[i][mt][4 * q + e];
                        const float t = fmaf(a, f[e], old);
                        sum[i][mt][4 * q + e] = t;
                        acc[i][mt][4 * q + e] = kCarry ? fmaf(a, f[e], old - t) * g[e] : 0.0f;
                    }
            }
    };
    // Q4_K: the finished slab's coefficient times sum products
    auto corrections = [&](int slab) {
        if constexpr (QT == kQ4_K) {
            const uint8_t* cp = cbuf + (slab & 1) * S::CB;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int lr = 64 * n + 32 * i + col;
                const mb_h8 Bh = *reinterpret_cast<const mb_h8*>(cp + lr * 16);
                const mb_h8 Bl = *reinterpret_cast<const mb_h8*>(cp + 64 * NW * 16 + lr * 16);
                const float f = reinterpret_cast<const float*>(cp + 64 * NW * 32)[lr];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const mb_h8 a = *reinterpret_cast<const mb_h8*>(
                        sbuf + (slab & 1) * S::SB + (mw * MT + mt) * 1024 + lane * 16);
                    mb_f16 t = mfma(a, Bl, mb_f16{});
                    t = mfma(a, Bh, t);
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][mt][r] = fmaf(f, t[r], acc[i][mt][r]);
                }
            }
        }
    };

    // Stage st computes on x and weight fragments in buffers st & 1, while x
    // of st + 1 is loaded, the weights of st + 1 (loaded during st - 1) are
    // decoded into the other buffer, and those of st + 2 are loaded.
    issue_x(st0);
    raw = pf_load_raw<QT>(wrow, 2 * st0 + wblk);
#pragma unroll
    for (int o = 0; o < 4; ++o) decode(o, st0 & 1, st0);
    raw = pf_load_raw<QT>(wrow, 2 * (st0 + 1) + wblk);
#pragma unroll 1
    for (int st = st0; st < st1; ++st) {
        // x of this stage and the next weights have landed, this stage's
        // fragments are written, and every wave is done with the other buffers
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (st + 1 < st1) issue_x(st + 1);
        // (past the last stage: a re-read of the last block, decoded but
        // never used)
        const int sn = st + 2 < st1 ? st + 2 : st1 - 1;
        const PfRaw<QT> next = pf_load_raw<QT>(wrow, 2 * sn + wblk);
        const int nb = (st & 1) ^ 1;

        const uint8_t* xs = xbuf + (st & 1) * S::XB + mw * MT * KST * 2048 + lane * 16;
        const uint8_t* ws = wbuf + (st & 1) * S::WB + 2 * n * KST * 1024 + lane * 16;
        const float* ds = reinterpret_cast<const float*>(dbuf + (st & 1) * S::DB) + 64 * n + col;
        auto xfrag = [&](int mt, int kl, int hl) {
            return *reinterpret_cast<const mb_h8*>(xs + ((mt * KST + kl) * 2 + hl) * 1024);
        };
#pragma unroll
        for (int bi = 0; bi < NBK; ++bi) {
            mb_h8 B[2][NK];
            float d[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                d[i] = ds[bi * 64 * NW + 32 * i];
#pragma unroll
                for (int p = 0; p < NK; ++p)
                    B[i][p] = *reinterpret_cast<const mb_h8*>(ws + (i * KST + NK * bi + p) * 1024);
            }
            // The wave's tiles one after the other: tile u's matrix-core
            // chain is issued with tile u - 1's block-scale FMAs, and a piece
            // of the next stage's decode, between its instructions (two tiles
            // of block sums live at a time).
            mb_f16 tmp[2];
            mb_h8 a[2][NK][2];
            auto read_x = [&](int mt) {
#pragma unroll
                for (int p = 0; p < NK; ++p)
#pragma unroll
                    for (int hl = 0; hl < 2; ++hl) a[mt & 1][p][hl] = xfrag(mt, NK * bi + p, hl);
            };
            auto scale_tile = [&](int u) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[u & 1][u >> 1][r] = fmaf(d[u & 1], tmp[u & 1][r], acc[u & 1][u >> 1][r]);
            };
            read_x(0);
#pragma unroll
            for (int u = 0; u < 2 * MT; ++u) {
                if ((u & 1) && (u >> 1) + 1 < MT) read_x((u >> 1) + 1);
                tmp[u & 1] = mb_f16{};
#pragma unroll
                for (int hl = 0; hl < 2; ++hl)
#pragma unroll
                    for (int p = 0; p < NK; ++p)
                        tmp[u & 1] = mfma(a[(u >> 1) & 1][p][hl], B[u & 1][p], tmp[u & 1]);
                if (u > 0) scale_tile(u - 1);
                constexpr int VN = 8 / NK;
                if (NK == 2 ? u >= 2 : u == 3) {
                    decode(NK == 2 ? 2 * bi + u - 2 : bi, nb, st + 1);
#pragma unroll
                    for (int p = 0; p < 2 * NK; ++p) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // matrix-core
                        __builtin_amdgcn_sched_group_barrier(0x002, VN + 3, 0);  // vector ALU
                    }
                } else {
#pragma unroll
                    for (int p = 0; p < 2 * NK; ++p) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, VN, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            scale_tile(2 * MT - 1);
        }
        raw = next;
        // (here, not after the barrier: the waves have drifted apart, and one
        // wave's flush runs beside another's matrix-core work)
        if ((st + 1) % kFlush == 0) {
            if ((st & 3) == 3) corrections(st >> 2);
            flush(st >> 2);
        }
    }

    const int tok0 = (mtile * TILES + mw * MT) * 32 + 4 * h;
    auto tok = [&](int mi, int r) { return tok0 + 32 * mi + 8 * (r >> 2) + (r & 3); };
    if (!whole && !j.pend) {
        // a split tile's partial sums, finished by pf_finish_kernel
        float* p = j.part + ((int64_t)(tile - j.tail0) * j.k_splits + split) * (kPfTile * 256) +
                   (int64_t)(tok0 - mtile * kPfTile) * 256 + 64 * n + col;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    p[(32 * mi + 8 * (r >> 2) + (r & 3)) * 256 + 32 * i] = sum[i][mi][r];
        return;
    }
    if constexpr (EPI == kPfSwiGLU) {
        const int row = nt_ * 32 * NW + 32 * n + col;
        if (row >= j.rows) return;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (tok(mi, r) < j.T)
                    j.y[(int64_t)tok(mi, r) * j.ld_y + row] =
                        swiglu_exact(sum[0][mi][r], sum[1][mi][r]);
    } else if constexpr (EPI == kPfAdd) {
        float* const y = whole ? j.y : j.part + (int64_t)split * j.T * j.rows;
        const int64_t ld = whole ? j.ld_y : j.rows;
        const bool accum = whole && j.accum;
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int row = nt_ * 64 * NW + 64 * n + 32 * i + col;
                if (row >= j.rows) continue;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (tok(mi, r) < j.T) {
                        float* p = y + (int64_t)tok(mi, r) * ld + row;
                        *p = accum ? *p + sum[i][mi][r] : sum[i][mi][r];
                    }
            }
    } else {
        // Rotated in registers: RoPE pairs are adjacent lanes (rows 2 p and
        // 2 p + 1, both of one segment).
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = nt_ * 64 * NW + 64 * n + 32 * i + col;
            int local;
            const int sgi = pf_segment(row, j.seg_end[0], j.seg_end[1], &local);
            const int half = j.head_dim / 2;
            const float2* csp = j.cs + (local % j.head_dim) / 2;
            const bool odd = col & 1;
            char* const cache = static_cast<char*>(sgi == 1 ? j.kc : j.vc);
#pragma unroll
            for (int mi = 0; mi < MT; ++mi)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float own = sum[i][mi][r], other = dpp_f32<0xB1>(own);
                    const int t = tok(mi, r);
                    if (t < j.T && row < j.rows) {
                        float v = own;
                        if (sgi < 2) {
                            const float2 cs = csp[(int64_t)t * half];
                            float a = odd ? other : own, b = odd ? own : other;
                            rot(a, b, cs.x, cs.y);
                            v = odd ? b : a;
                        }
                        if (sgi == 0) {
                            j.y[(int64_t)t * j.ld_y + local] = v;
                        } else {
                            const int ps = j.pos[t];
                            const int64_t ci = (int64_t)ps * j.kv_dim + local;
                            if (ps >= 0 && ps < j.max_ctx) {
                                if (j.kv_f16)
                                    *reinterpret_cast<uint16_t*>(cache + 2 * ci) = f2h(v);
                                else
                                    *reinterpret_cast<float*>(cache + 4 * ci) = v;
                            }
                        }
                    }
                }
        }
    }
}

// The split tiles' partial sums, added in split order, and their epilogue:
// grid (tail tiles x 32), each workgroup 4 tokens of a tile, a lane two rows
// of one token (kPfSwiGLU: a gate row and its up row; else a RoPE pair).
template <int EPI>
__global__ __launch_bounds__(256) void pf_finish_kernel(PfJob j) {
    const int tl = blockIdx.x >> 5, tile = j.tail0 + tl;
    const int mtile = tile % j.n_mt, nt = tile / j.n_mt;
    const int pr = threadIdx.x & 127;
    const int l0 = EPI == kPfSwiGLU ? 64 * (pr >> 5) + (pr & 31) : 2 * pr;
    const int l1 = EPI == kPfSwiGLU ? l0 + 32 : l0 + 1;
    const int row = EPI == kPfSwiGLU ? nt * 128 + 32 * (pr >> 5) + (pr & 31) : nt * 256 + l0;
    if (row >= j.rows) return;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int lt = (blockIdx.x & 31) * 4 + 2 * k + (threadIdx.x >> 7);
        const int t = mtile * kPfTile + lt;
        if (t >= j.T) return;
        const float* p = j.part + (int64_t)tl * j.k_splits * (kPfTile * 256) + lt * 256;
        float a = 0.0f, b = 0.0f;
#pragma unroll 4
        for (int s = 0; s < j.k_splits; ++s) {
            a += p[(int64_t)s * (kPfTile * 256) + l0];
            b += p[(int64_t)s * (kPfTile * 256) + l1];
        }
        if constexpr (EPI == kPfSwiGLU) {
            j.y[(int64_t)t * j.ld_y + row] = swiglu_exact(a, b);
        } else if constexpr (EPI == kPfAdd) {
            float* y = j.y + (int64_t)t * j.ld_y + row;
            y[0] = j.accum ? y[0] + a : a;
            if (row + 1 < j.rows) y[1] = j.accum ? y[1] + b : b;
        } else {
            int local;
            const int sgi = pf_segment(row, j.seg_end[0], j.seg_end[1], &local);
            if (sgi < 2) {
                const float2 cs = j.cs[(int64_t)t * (j.head_dim / 2) + (local % j.head_dim) / 2];
                rot(a, b, cs.x, cs.y);
            }
            if (sgi == 0) {
                float* y = j.y + (int64_t)t * j.ld_y + local;
                y[0] = a;
                y[1] = b;
                continue;
            }
            const int ps = j.pos[t];
            if (ps < 0 || ps >= j.max_ctx) continue;
            const int64_t ci = (int64_t)ps * j.kv_dim + local;
            char* cp = static_cast<char*>(sgi == 1 ? j.kc : j.vc);
            if (j.kv_f16) {
                uint16_t* c = reinterpret_cast<uint16_t*>(cp) + ci;
                c[0] = f2h(a);
                c[1] = f2h(b);
            } else {
                float* c = reinterpret_cast<float*>(cp) + ci;
                c[0] = a;
                c[1] = b;
            }
        }
    }
}

// Tiles run in rounds of one workgroup per CU.  The tiles left over from the
// last whole round are split over the columns as far as that round has CUs
// for (a 1000-token prompt's gate / up product at Llama-3-8B widths: 896
// tiles, 3 rounds of 256 and 128 tiles in two halves).  A residual add whose
// tiles all fit in one round leaves its splits' sums pending instead, merged
// by the next preparation's pass over the residual stream.
template <int QT, int EPI>
int pf_launch(PfJob& j, size_t part_bytes, hipStream_t stream) {
    using S = PfShape<QT>;
    constexpr int NW = S::NW;
    const int per_tile = EPI == kPfSwiGLU ? 32 * NW : 64 * NW;
    j.n_nt = (j.rows + per_tile - 1) / per_tile;
    j.n_mt = (j.T + kPfTile - 1) / kPfTile;
    const int tiles = j.n_nt * j.n_mt, rounds = tiles / kPfTarget;
    const int tail = tiles - rounds * kPfTarget;
    int k = tail > 0 ? kPfTarget / tail : 1;
    if (k > j.n_slabs) k = j.n_slabs;
    j.slabs_per_split = (j.n_slabs + k - 1) / k;
    j.k_splits = (j.n_slabs + j.slabs_per_split - 1) / j.slabs_per_split;
    if (rounds > 0 || j.k_splits == 1) j.pend = 0;
    j.tail0 = rounds * kPfTarget;
    j.full_per_xcd = j.tail0 / 8;
    j.tail_items = tail * j.k_splits;
    j.tail_per_xcd = (j.tail_items + 7) / 8;
    const size_t tile_rows = j.pend ? (size_t)j.T * j.rows : (size_t)tail * kPfTile * 256;
    if (j.k_splits > 1 && j.k_splits * tile_rows * sizeof(float) > part_bytes)
        return JINF_HIP_ERR_INVALID;  // (the buffer holds kPfTarget split tiles)
    const int rc = launch(pf_matmul_kernel<QT, EPI>, dim3(8 * (j.full_per_xcd + j.tail_per_xcd)),
                          dim3(512), S::LDS, stream, j);
    if (rc != JINF_HIP_OK || j.k_splits == 1 || tail == 0 || j.pend) return rc;
    return launch(pf_finish_kernel<EPI>, dim3((unsigned)(32 * tail)), dim3(256), 0, stream, j);
}

template <int EPI>
int pf_dispatch(int qtype, PfJob& j, const PfBuf& b, hipStream_t stream) {
    switch (qtype) {
        case kQ4_0: return pf_launch<kQ4_0, EPI>(j, b.part_bytes, stream);
        case kQ8_0: return pf_launch<kQ8_0, EPI>(j, b.part_bytes, stream);
        case kQ4_K: return pf_launch<kQ4_K, EPI>(j, b.part_bytes, stream);
        case kQ6_K: return pf_launch<kQ6_K, EPI>(j, b.part_bytes, stream);
        default: return JINF_HIP_ERR_INVALID;
    }
}

// Fields common to every product; JINF_HIP_ERR_INVALID for shapes and
// alignments the kernel does not take.
int pf_job(PfJob& j, const PfBuf& b, int qtype, int T, int rows, int cols, float* y, int ld_y,
           const void* w0, const void* w1, const void* w2) {
    int e, bytes;
    switch (qtype) {
        case kQ4_0: e = 32; bytes = 18; break;
        case kQ8_0: e = 32; bytes = 34; break;
        case kQ4_K: e = 256; bytes = 144; break;
        case kQ6_K: e = 256; bytes = 210; break;
        default: return JINF_HIP_ERR_INVALID;
    }
    if (T <= 0 || T > b.rows || rows <= 0 || cols <= 0 || cols % kMbCols != 0 || !y)
        return JINF_HIP_ERR_INVALID;
    for (const void* w : {w0, w1, w2})
        if (!w || !aligned(w, 16)) return JINF_HIP_ERR_INVALID;
    j.rows = rows;
    j.n_slabs = cols / kMbCols;
    j.T = T;
    j.W[0] = static_cast<const uint8_t*>(w0);
    j.W[1] = static_cast<const uint8_t*>(w1);
    j.W[2] = static_cast<const uint8_t*>(w2);
    j.seg_end[0] = j.seg_end[1] = j.seg_end[2] = rows;
    j.row_bytes = (int64_t)(cols / e) * bytes;
    j.rec = b.rec;
    j.xs = b.xs;
    j.y = y;
    j.ld_y = ld_y;
    j.part = b.part;
    return JINF_HIP_OK;
}

}  // namespace

size_t pf_rec_bytes(int rows, int cols) { return (size_t)(rows / 32) * (cols / kMbCols) * kPfRec; }

// At most kPfTarget split tiles, each holding kPfTile x 256 partial sums.
size_t pf_part_bytes() { return (size_t)kPfTarget * kPfTile * 256 * sizeof(float); }

int pf_rope_table(const PfBuf& b, const int32_t* positions, int T, int head_dim, float freq_base,
                  hipStream_t stream) {
    RopeTheta th;
    theta_table(th, head_dim, freq_base);
    const int half = head_dim / 2;
    return launch(pf_rope_table_kernel, dim3((unsigned)((T * half + 255) / 256)), dim3(256), 0,
                  stream, b.cs, positions, T * half, half, th);
}

int pf_prepare(const PfBuf& b, float* x, int ld_x, int T, int cols, const void* norm_w,
               int norm_type, float eps, PfPend* pend, hipStream_t stream) {
    const int f16 = norm_w && norm_type == JINF_HIP_F16;
    const int k = pend ? pend->k : 0;
    const unsigned tokens = (unsigned)((T + kPfTile - 1) / kPfTile * kPfTile);
    const int ng = (cols / 8 + 255) / 256;
    if (ng > 16) return JINF_HIP_ERR_INVALID;  // (the batch takes at most 32768 columns)
    auto* kern = ng <= 1   ? pf_prepare_kernel<1>
                 : ng <= 2 ? pf_prepare_kernel<2>
                 : ng <= 4 ? pf_prepare_kernel<4>
                 : ng <= 8 ? pf_prepare_kernel<8>
                           : pf_prepare_kernel<16>;
    const int rc = launch(kern, dim3(tokens), dim3(256), 0, stream, x, ld_x, cols, T,
                          static_cast<const float*>(b.part), k, (int64_t)T * cols, norm_w, f16, eps,
                          b.xs, b.rec);
    if (rc == JINF_HIP_OK && pend) pend->k = 0;
    return rc;
}

int pf_merge(const PfBuf& b, float* x, int ld_x, int T, int cols, PfPend* pend,
             hipStream_t stream) {
    if (pend->k == 0) return JINF_HIP_OK;
    const int rc = launch(pf_merge_kernel, dim3((unsigned)((cols / 8 + 255) / 256), (unsigned)T),
                          dim3(256), 0, stream, x, ld_x, cols, static_cast<const float*>(b.part),
                          pend->k, (int64_t)T * cols);
    pend->k = 0;
    return rc;
}

int pf_matmul(const PfBuf& b, const void* w, int qtype, int T, int rows, int cols, float* y,
              int ld_y, bool accum, PfPend* pend, hipStream_t stream) {
    PfJob j{};
    int rc = pf_job(j, b, qtype, T, rows, cols, y, ld_y, w, w, w);
    if (rc != JINF_HIP_OK) return rc;
    j.accum = accum;
    j.pend = accum && pend;
    rc = pf_dispatch<kPfAdd>(qtype, j, b, stream);
    if (pend) pend->k = rc == JINF_HIP_OK && j.pend ? j.k_splits : 0;
    return rc;
}

int pf_swiglu(const PfBuf& b, const void* w_gate, const void* w_up, int qtype, int T, int n_ff,
              int cols, float* y, int ld_y, hipStream_t stream) {
    PfJob j{};
    const int rc = pf_job(j, b, qtype, T, n_ff, cols, y, ld_y, w_gate, w_up, w_gate);
    if (rc != JINF_HIP_OK) return rc;
    return pf_dispatch<kPfSwiGLU>(qtype, j, b, stream);
}

int pf_qkv(const PfBuf& b, const void* wq, const void* wk, const void* wv, int qtype, int T,
           int cols, float* q, int ld_q, void* kc, void* vc, int kv_type,
           const int32_t* positions, int max_ctx, int head_dim, int n_heads, int n_heads_kv,
           hipStream_t stream) {
    const int qd = n_heads * head_dim, kvd = n_heads_kv * head_dim;
    const void* first = wq ? wq : wk ? wk : wv;
    PfJob j{};
    const int len[3] = {wq ? qd : 0, wk ? kvd : 0, wv ? kvd : 0};
    const int rc = pf_job(j, b, qtype, T, len[0] + len[1] + len[2], cols, q, ld_q, wq ? wq : first,
                          wk ? wk : first, wv ? wv : first);
    if (rc != JINF_HIP_OK) return rc;
    j.seg_end[0] = len[0];
    j.seg_end[1] = len[0] + len[1];
    j.cs = b.cs;
    j.pos = positions;
    j.kc = kc;
    j.vc = vc;
    j.kv_f16 = kv_type == JINF_HIP_F16;
    j.kv_dim = kvd;
    j.head_dim = head_dim;
    j.max_ctx = max_ctx;
    return pf_dispatch<kPfQKV>(qtype, j, b, stream);
}

}  // namespace jinf
