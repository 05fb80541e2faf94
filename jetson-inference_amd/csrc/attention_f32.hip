// Decode attention over an fp32 KV cache, contexts split over workgroups
// (reference cuda/attention_kernel.cu:25-96; the cache type its engine keeps).
//
// What bounds it: the K and V rows' bytes, and at batch 1 having enough of
// them in flight.  A head's whole context streamed through one workgroup takes
// 94 us (32 heads, 4096 positions: 0.36 TB/s; 17.0 us here, the error against
// fp64 3.5e-7 -> 2.1e-7).  Here a workgroup takes one kv head's whole query group, so
// each row is read once, and a chunk of the context; its 8 waves take 16
// positions at a time and each has the 16 K and 16 V rows' loads (16 KiB at
// head_dim 128) in flight before any arithmetic.
//   - Scores: LPP lanes per position hold a slice of the K row and of every
//     query head, partial dots are reduced with DPP.
//   - Softmax: online per wave over its 16-position tiles, in registers.
//   - P V: half a wave per V row (16-byte loads), the probabilities read from
//     the lanes that hold them; the two halves are added at the end.
//   - The waves merge through LDS, the chunks as the fp16 kernel's do.
#include <hip/hip_runtime.h>
#include <math.h>

#include <type_traits>

#include "attention_device.h"
#include "jinf_device.h"
#include "jinf_host.h"

namespace jinf {
namespace {

constexpr int kFwWaves = 8;
constexpr int kFwTile = 16;  // positions per wave and step

// max / sum over the lanes l, l ^ LPP, l ^ 2 LPP, ... (LPP a power of two):
// lanes of one position hold the same value
template <int LPP>
__device__ __forceinline__ float across_max(float v) {
    if constexpr (LPP <= 4) v = fmaxf(v, __shfl_xor(v, 4, kWave));
    if constexpr (LPP <= 8) v = fmaxf(v, dpp_f32<0x128>(v));  // row_ror:8
    v = fmaxf(v, __shfl_xor(v, 16, kWave));
    return xor32_max(v);
}
template <int LPP>
__device__ __forceinline__ float across_sum(float v) {
    if constexpr (LPP <= 4) v += __shfl_xor(v, 4, kWave);
    if constexpr (LPP <= 8) v += dpp_f32<0x128>(v);
    v += __shfl_xor(v, 16, kWave);
    return xor32_sum(v);
}

// grid (n_heads / G, n_seq, chunks), 512 threads.
template <int HD, int G, bool MERGE>
__global__ __launch_bounds__(64 * kFwWaves, 2) void attn_f32_kernel(
    const int32_t* __restrict__ lens, int n_past, int chunk, int group,
    const float* __restrict__ kc, const float* __restrict__ vc, int64_t ld_pos, int64_t ld_seq,
    const float* __restrict__ q, int64_t ld_q, int n_heads, float scale, float* __restrict__ out,
    int64_t ld_out, float* __restrict__ ws, unsigned* __restrict__ counters) {
    constexpr int LPP = G * HD / 64 > HD / 16 ? G * HD / 64 : HD / 16;  // lanes per position
    constexpr int DPQ = HD / LPP;              // dims per lane: G DPQ <= 64 q registers
    constexpr int PPP = kWave / LPP;           // positions per pass
    constexpr int NP = kFwTile / PPP;          // passes per tile
    constexpr int VL = HD / 4;                 // lanes per V row
    constexpr int VR = kWave / VL;             // V rows per load
    constexpr int NV = kFwTile / VR;           // V loads per tile
    constexpr int MS = HD + 2;
    static_assert(LPP >= 4 && LPP <= 16 && DPQ % 4 == 0 && NP >= 1, "lane layout");
    extern __shared__ __attribute__((aligned(16))) uint8_t fw_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x & (kWave - 1);
    const int s = blockIdx.y, cix = blockIdx.z, nch = gridDim.z;
    const int h0 = blockIdx.x * G;
    const int j = h0 / group;
    const int len = lens ? min(max(lens[s], 0), n_past) : n_past;
    const int c0 = cix * chunk, c1 = min(c0 + chunk, len);
    // chunk 0 always runs (an empty context writes zeros)
    if (cix > 0 && c0 >= len) return;
    const int used = (len + chunk - 1) / chunk;
    const float* kb = kc + (int64_t)s * ld_seq + (int64_t)j * HD;
    const float* vb = vc + (int64_t)s * ld_seq + (int64_t)j * HD;
    const int sub = lane % LPP, pl = lane / LPP;    // slice, position of the pass
    const int vr = lane / VL, vd = 4 * (lane % VL); // V row of the load, dims

    float4 kv[NP][DPQ / 4], vv[NV];
    // rows past the chunk's end re-read its last one (their probability is 0)
    auto load = [&](int t0) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int pos = min(t0 + p * PPP + pl, c1 - 1);
            const float4* kp = reinterpret_cast<const float4*>(kb + (int64_t)pos * ld_pos + sub * DPQ);
#pragma unroll
            for (int c = 0; c < DPQ / 4; ++c) kv[p][c] = kp[c];
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int pos = min(t0 + VR * i + vr, c1 - 1);
            vv[i] = *reinterpret_cast<const float4*>(vb + (int64_t)pos * ld_pos + vd);
        }
    };
    const int tfirst = c0 + wave * kFwTile;
    if (tfirst < c1) load(tfirst);

    float qv[G][DPQ];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float4* qp = reinterpret_cast<const float4*>(
            q + (int64_t)s * ld_q + (int64_t)(h0 + g) * HD + sub * DPQ);
#pragma unroll
        for (int c = 0; c < DPQ / 4; ++c) {
            const float4 x = qp[c];
            qv[g][4 * c] = x.x; qv[g][4 * c + 1] = x.y; qv[g][4 * c + 2] = x.z; qv[g][4 * c + 3] = x.w;
        }
    }
    float m[G], l[G], acc[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[g][e] = 0.0f;
    }
    if (tfirst < c1)
    for (int t0 = tfirst;;) {
        // scores of the tile: sc[g][p] for position t0 + p PPP + pl
        float pr[G][NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const bool live = t0 + p * PPP + pl < c1;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float d = 0.0f;
#pragma unroll
                for (int c = 0; c < DPQ / 4; ++c) {
                    d = fmaf(qv[g][4 * c], kv[p][c].x, d);
                    d = fmaf(qv[g][4 * c + 1], kv[p][c].y, d);
                    d = fmaf(qv[g][4 * c + 2], kv[p][c].z, d);
                    d = fmaf(qv[g][4 * c + 3], kv[p][c].w, d);
                }
                d += dpp_f32<0xB1>(d);
                d += dpp_f32<0x4E>(d);
                if constexpr (LPP >= 8) d += __shfl_xor(d, 4, kWave);
                if constexpr (LPP >= 16) d += dpp_f32<0x128>(d);
                pr[g][p] = live ? d * scale : -INFINITY;
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float tm = pr[g][0];
#pragma unroll
            for (int p = 1; p < NP; ++p) tm = fmaxf(tm, pr[g][p]);
            const float mn = fmaxf(m[g], across_max<LPP>(tm));
            const float ms = softmax_ref(mn);
            const float corr = exp_neg_fast(m[g] - ms);
            float ts = 0.0f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                pr[g][p] = exp_neg_fast(pr[g][p] - ms);
                ts += pr[g][p];
            }
            l[g] = fmaf(l[g], corr, across_sum<LPP>(ts));
            m[g] = mn;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[g][e] *= corr;
        }
        // P V: load i holds rows VR i + vr; row r's probability sits in pass
        // r / PPP, lanes (r % PPP) LPP ..
#pragma unroll
        for (int i = 0; i < NV; ++i) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float p = 0.0f;
#pragma unroll
                for (int u = 0; u < VR; ++u) {
                    const int r = VR * i + u;
                    const float x = __int_as_float(__builtin_amdgcn_readlane(
                        __float_as_int(pr[g][r / PPP]), (r % PPP) * LPP));
                    p = u == 0 || vr == u ? x : p;
                }
                acc[g][0] = fmaf(p, vv[i].x, acc[g][0]);
                acc[g][1] = fmaf(p, vv[i].y, acc[g][1]);
                acc[g][2] = fmaf(p, vv[i].z, acc[g][2]);
                acc[g][3] = fmaf(p, vv[i].w, acc[g][3]);
            }
        }
        t0 += kFwWaves * kFwTile;
        if (t0 >= c1) break;
        load(t0);
    }

    // the lanes' V rows, then the waves (in wave order) through LDS
    float* mg = reinterpret_cast<float*>(fw_lds);  // [waves][G][MS]
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (VR >= 4) acc[g][e] += __shfl_xor(acc[g][e], 16, kWave);
            acc[g][e] = xor32_sum(acc[g][e]);
        }
        float* r = mg + (wave * G + g) * MS;
        if (lane < VL) {
            // (MS is even: 8-byte aligned)
            reinterpret_cast<float2*>(r + vd)[0] = make_float2(acc[g][0], acc[g][1]);
            reinterpret_cast<float2*>(r + vd)[1] = make_float2(acc[g][2], acc[g][3]);
        }
        if (lane == 0) {
            r[HD] = m[g];
            r[HD + 1] = l[g];
        }
    }
    __syncthreads();
    const bool direct = !ws || used <= 1;
    for (int idx = threadIdx.x; idx < G * HD; idx += 64 * kFwWaves) {
        const int g = idx / HD, d = idx % HD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kFwWaves; ++w) M = fmaxf(M, mg[(w * G + g) * MS + HD]);
        const float Ms = softmax_ref(M);
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int w = 0; w < kFwWaves; ++w) {
            const float* e = mg + (w * G + g) * MS;
            const float f = exp_neg_fast(e[HD] - Ms);  // idle waves: 0
            num = fmaf(f, e[d], num);
            den = fmaf(f, e[HD + 1], den);
        }
        if (direct) {
            out[(int64_t)s * ld_out + (int64_t)(h0 + g) * HD + d] = len > 0 ? num / den : 0.0f;
        } else {
            float* rec = ws + (((int64_t)s * n_heads + h0 + g) * nch + cix) * MS;
            if constexpr (MERGE) {
                rec_store(rec + d, num);
                if (d == 0) {
                    rec_store(rec + HD, M);
                    rec_store(rec + HD + 1, den);
                }
            } else {
                rec[d] = num;
                if (d == 0) {
                    rec[HD] = M;
                    rec[HD + 1] = den;
                }
            }
        }
    }
    if constexpr (MERGE) {
        if (!direct)
            am_merge_last<HD>(out, ld_out, ws, counters, s, n_heads, h0, G, nch, used, fw_lds);
    }
}

template <int HD, int G>
int fw_launch(float* out, int64_t ld_out, const float* q, int64_t ld_q, const float* k,
              const float* v, int64_t ld_pos, int64_t ld_seq, const int32_t* lens, int n_past,
              int n_seq, int n_heads, int group, int chunk, int nch, float scale, float* ws,
              unsigned* counters, hipStream_t stream) {
    // the waves' records; the in-kernel merge's 16 floats per chunk (+ 8)
    size_t shmem = (size_t)kFwWaves * G * (HD + 2) * 4;
    const size_t merge = ((size_t)nch * 16 + 8) * 4;
    if (counters && merge > shmem) shmem = merge;
    auto* kern = counters ? attn_f32_kernel<HD, G, true> : attn_f32_kernel<HD, G, false>;
    return launch(kern, dim3(n_heads / G, n_seq, nch), dim3(64 * kFwWaves), shmem, stream, lens,
                  n_past, chunk, group, k, v, ld_pos, ld_seq, q, ld_q, n_heads, scale, out, ld_out,
                  ws, counters);
}

}  // namespace

int attn_f32_launch(float* out, int64_t ld_out, const float* q, int64_t ld_q, const void* k,
                    const void* v, int64_t ld_pos, int64_t ld_seq, const int32_t* lens,
                    int n_past, int n_seq, int head_dim, int n_heads, int group, int G, int chunk,
                    int nch, float scale, float* ws, unsigned* counters, hipStream_t stream) {
    auto go = [&](auto hd, auto g) {
        return fw_launch<decltype(hd)::value, decltype(g)::value>(
            out, ld_out, q, ld_q, static_cast<const float*>(k), static_cast<const float*>(v),
            ld_pos, ld_seq, lens, n_past, n_seq, n_heads, group, chunk, nch, scale, ws, counters,
            stream);
    };
    auto pick = [&](auto hd) {
        switch (G) {
            case 8: return go(hd, std::integral_constant<int, 8>{});
            case 4: return go(hd, std::integral_constant<int, 4>{});
            case 2: return go(hd, std::integral_constant<int, 2>{});
            default: return go(hd, std::integral_constant<int, 1>{});
        }
    };
    return head_dim == 64 ? pick(std::integral_constant<int, 64>{})
                          : pick(std::integral_constant<int, 128>{});
}

}  // namespace jinf
