// Causal GQA attention of many tokens of one prompt against its fp16 KV cache
// (reference cuda/attention_kernel.cu:25-96, called once per token): row t
// attends to the positions below lens[t].
//
// Arithmetic: the fp16 matrix-core kernel's of attention.hip.  Scores are
// K Q' with q scale split into fp16 hi + lo, the probabilities (times 2^15)
// likewise in P' V, so every product keeps about 22 bits; the softmax state
// is fp32 and online over 64-position tiles.
//
// What bounds it: run per row (the decode kernel with one work item per token
// and kv head), every token re-reads its whole context and half the
// matrix-core columns are empty at 4 query heads per kv head: 252 us per
// layer for a 1000-token prompt at 32 / 8 heads x 128.  Here a workgroup
// takes 64 (token, head) rows of one kv head, 64 / G consecutive tokens of G
// heads, and its 4 waves share each K / V tile from LDS, 16 rows a wave (two
// groups of 8 rows x {hi, lo} columns).  No cross-wave merge is needed, and
// the tiles are double-buffered: 64 KiB at head_dim 128, two workgroups per
// CU.  Later tokens have longer contexts, so their workgroups start first.
//
// Few tokens far into a context give few workgroups with many tiles each (65
// tokens at position 8000: 40 of 127).  Their contexts are split over the
// grid's third dimension; each chunk leaves {O, m, l} records like the decode
// kernel's, merged by its combine launch.  Prompts of 4 layers of 4096 /
// 14336, at position 8000: 65 tokens 1919 -> 1125 us, 128 2011 -> 1249, 256
// 2490 -> 1899, 1000 unchanged; 2 tokens 1810 -> 958.  (Twice the workgroups
// aimed for: 1180, 1315, 1956; chunks of 128: 1120, 1258, 1897, 2 tokens 1001.)
#include <hip/hip_runtime.h>
#include <math.h>

#include "attention_device.h"
#include "jinf_device.h"
#include "jinf_host.h"
#include "jinf/kernels_ext.h"
#include "prefill_internal.h"

namespace jinf {
namespace {

typedef _Float16 pa_h4 __attribute__((ext_vector_type(4)));
typedef _Float16 pa_h8 __attribute__((ext_vector_type(8)));
typedef float pa_f4 __attribute__((ext_vector_type(4)));
typedef short pa_tr4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) pa_tr4 pa_lds_tr4;

constexpr int kPaTile = 64;            // positions per tile
constexpr int kPaRows = 64;            // (token, head) rows per workgroup
constexpr float kPaPScale = 32768.0f;  // 2^15: probabilities in fp16's normal range
constexpr int kPaTarget = 512;         // workgroups (two per CU) that splits aim for
constexpr int kPaChunkMin = 256;       // positions per chunk, at least

__device__ __forceinline__ pa_h8 pa_cat(pa_h4 a, pa_h4 b) {
    return pa_h8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// grid (token tiles, n_heads / G, chunks), 256 threads; group = query heads
// per kv head (a multiple of G).  SPLIT: chunks of `chunk` positions (a
// multiple of the tile); a row whose context fits in one is written directly,
// else its chunks' records go to ws[token][head][chunk].
template <int HD, bool SPLIT>
__global__ __launch_bounds__(256, 2) void pf_attention_kernel(
    const int32_t* __restrict__ lens, int T, int n_ctx, int G, int group,
    const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, int64_t ld_pos,
    const float* __restrict__ q, int64_t ld_q, float scale, float* __restrict__ out,
    int64_t ld_out, int chunk, int n_heads, float* __restrict__ ws) {
    constexpr int KS = HD / 16;       // 4-dim groups of q per lane
    constexpr int DPG = HD / 4;       // dims per lane group in the score product
    constexpr int KLD = DPG / 8;      // 32-deep k-steps of the score product
    constexpr int NB = HD / 16;       // 16-dim blocks of the output
    constexpr int VCH = HD / 8;       // 16-byte chunks per row
    constexpr int LD = kPaTile * VCH / 256;  // loads per lane per tile (K or V)
    constexpr int PITCH = HD * 2;
    constexpr int BUF = 2 * kPaTile * PITCH;  // K tile, V tile
    extern __shared__ __attribute__((aligned(16))) uint8_t pa_lds[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid & (kWave - 1);
    const int col = lane & 15, lg = lane >> 4;
    const bool lo_col = col >= 8;
    const int TQ = kPaRows / G;
    const int qt = gridDim.x - 1 - blockIdx.x;  // longest contexts first
    const int tok_base = qt * TQ;
    const int h0 = blockIdx.y * G;
    const int j = h0 / group;

    // row of column slot s of the wave's group g: 16 wave + 8 g + s -> (token, head)
    auto row_of = [&](int g, int s, int& tok, int& head) {
        const int idx = 16 * wave + 8 * g + s;
        tok = tok_base + idx / G;
        head = h0 + idx % G;
    };
    int lim[2];      // positions the lane's column attends to
    int wlim = 0;    // the most of any column of the wave
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        int tok, head;
        row_of(g, col & 7, tok, head);
        lim[g] = tok < T ? min(max(lens[tok], 0), n_ctx) : 0;
        wlim = max(wlim, lim[g]);
    }
    // the longest and shortest context of the workgroup's tokens
    int wg_lim = 0, wg_min = n_ctx;
    for (int i = 0; i < TQ; ++i) {
        const int tok = tok_base + i;
        if (tok >= T) break;
        const int l = min(max(lens[tok], 0), n_ctx);
        wg_lim = max(wg_lim, l);
        wg_min = min(wg_min, l);
    }
#pragma unroll
    for (int o = 1; o < kWave; o *= 2) wlim = max(wlim, __shfl_xor(wlim, o, kWave));
    wlim = __builtin_amdgcn_readfirstlane(wlim);
    // rows of V with a non-finite value in the current tile (see below)
    __shared__ unsigned bad_rows[2][2];
    if (tid < 4) bad_rows[tid >> 1][tid & 1] = 0u;

    // the workgroup's positions: c0 .. c1
    const int c0 = SPLIT ? (int)blockIdx.z * chunk : 0;
    const int c1 = SPLIT ? min(wg_lim, c0 + chunk) : wg_lim;
    if (SPLIT && c0 > 0 && c0 >= wg_lim) return;  // (before any barrier, workgroup-uniform)

    const uint32_t rowb = (uint32_t)ld_pos * 2;
    const int nrec = (int)((uint32_t)wg_lim * rowb);
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(kc + (int64_t)j * HD), (short)0, nrec, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(vc + (int64_t)j * HD), (short)0, nrec, 0x00020000);
    // LDS layout of a tile as in the decode kernel: K slot (row r, p) holds
    // chunk p ^ kswz(r), V slot (r, p) chunk p ^ 2 (r & 3)
    auto kswz = [](int r) { return HD == 128 ? (r & 15) : ((r >> 1) & 7); };
    uint32_t koff[LD], voff[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const int slot = (wave * LD + i) * kWave + lane;
        const int row = slot / VCH;
        koff[i] = (uint32_t)row * rowb + 16u * (uint32_t)((slot % VCH) ^ kswz(row));
        voff[i] = (uint32_t)row * rowb + 16u * (uint32_t)((slot % VCH) ^ (2 * (row & 3)));
    }
    auto load_tile = [&](int t0, int buf) {
        uint8_t* kb = pa_lds + buf * BUF;
        const uint32_t so = (uint32_t)t0 * rowb;
#pragma unroll
        for (int i = 0; i < LD; ++i) lds_load16_buf(krs, koff[i], so, kb + 1024 * (wave * LD + i));
#pragma unroll
        for (int i = 0; i < LD; ++i)
            lds_load16_buf(vrs, voff[i], so, kb + kPaTile * PITCH + 1024 * (wave * LD + i));
    };
    if (c0 < c1) load_tile(c0, 0);

    // q scale as fp16 hi / lo B fragments: the lane's 8 dims DPG lg + 8 u .. + 7
    pa_h8 qf[2][KLD];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        int tok, head;
        row_of(g, col & 7, tok, head);
        const bool live = tok < T;
        const float4* qp = reinterpret_cast<const float4*>(
            q + (int64_t)(live ? tok : 0) * ld_q + (int64_t)head * HD + DPG * lg);
        const float qs = live ? scale : 0.0f;
        pa_h4 f[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float4 v = qp[ks];
            const float x[4] = {v.x * qs, v.y * qs, v.z * qs, v.w * qs};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const _Float16 hi = (_Float16)x[i];
                f[ks][i] = lo_col ? (_Float16)(x[i] - (float)hi) : hi;
            }
        }
#pragma unroll
        for (int u = 0; u < KLD; ++u) qf[g][u] = pa_cat(f[2 * u], f[2 * u + 1]);
    }

    float m[2] = {-INFINITY, -INFINITY}, lsum[2] = {0.0f, 0.0f};
    bool poison[2] = {false, false};
    pa_f4 O[2][NB];
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int n = 0; n < NB; ++n) O[g][n] = pa_f4{0.f, 0.f, 0.f, 0.f};

    int buf = 0;
    for (int t0 = c0; t0 < c1; t0 += kPaTile, buf ^= 1) {
        // this tile has landed for every wave, and every wave has finished
        // with the other buffer
        __builtin_amdgcn_s_waitcnt(waitcnt_vm<0>());
        __syncthreads();
        if (t0 + kPaTile < c1) load_tile(t0 + kPaTile, buf ^ 1);
        // A tile in which some row's context ends holds later tokens' V rows.
        // Their probabilities are 0, but 0 times a non-finite value is not:
        // such values are cleared in LDS, and rows that do attend to one give
        // NaN at the end.  (Scanning costs those one or two tiles per
        // workgroup a barrier and 4 LDS reads a lane.)
        unsigned long long bad = 0;
        if (t0 + kPaTile > wg_min) {
            uint8_t* vt = pa_lds + buf * BUF + kPaTile * PITCH;
#pragma unroll 1
            for (int i = 0; i < LD; ++i) {
                const int at = 16 * (256 * i + tid);
                uint4 w = *reinterpret_cast<const uint4*>(vt + at);
                uint32_t x[4] = {w.x, w.y, w.z, w.w};
                bool nf = false;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if ((x[e] & 0x7C00u) == 0x7C00u) nf = true, x[e] &= 0xFFFF0000u;
                    if ((x[e] & 0x7C000000u) == 0x7C000000u) nf = true, x[e] &= 0xFFFFu;
                }
                if (nf) {
                    *reinterpret_cast<uint4*>(vt + at) = make_uint4(x[0], x[1], x[2], x[3]);
                    atomicOr(&bad_rows[buf][(at / PITCH) >> 5], 1u << ((at / PITCH) & 31));
                }
            }
            __syncthreads();
            bad = bad_rows[buf][0] | ((unsigned long long)bad_rows[buf][1] << 32);
            if (tid < 2) bad_rows[buf ^ 1][tid] = 0u;  // the next tile's (read before this barrier)
        }
        if (t0 >= wlim) continue;  // wave-uniform: none of its rows reaches here
        const uint8_t* kst = pa_lds + buf * BUF;
        const uint8_t* vst = kst + kPaTile * PITCH;
        pa_f4 S[2][4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int r = 16 * b + col;
            S[0][b] = S[1][b] = pa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < KLD; ++u) {
                const int c = (DPG * lg) / 8 + u;
                const pa_h8 kf = *reinterpret_cast<const pa_h8*>(kst + r * PITCH + 16 * (c ^ kswz(r)));
#pragma unroll
                for (int g = 0; g < 2; ++g)
                    S[g][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[g][u], S[g][b], 0, 0, 0);
            }
        }
        pa_h4 P[2][4];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            // hi + lo columns, mask, tile max over the column's four lane groups
            float tmax = -INFINITY;
            const int left = lim[g] - t0 - 4 * lg;
            if (bad) {
                const int live = min(max(lim[g] - t0, 0), kPaTile);
                if (live > 0 && (bad << (kPaTile - live)) != 0) poison[g] = true;
            }
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = S[g][b][r] + dpp_f32<0x128>(S[g][b][r]);  // row_ror:8
                    const float vm = 16 * b + r < left ? v : -INFINITY;
                    S[g][b][r] = vm;
                    tmax = fmaxf(tmax, vm);
                }
            tmax = fmaxf(tmax, __shfl_xor(tmax, 16, kWave));
            tmax = xor32_max(tmax);
            const float mn = fmaxf(m[g], tmax);
            // a column with no live position yet has mn = -inf: subtract 0, so
            // that its probabilities exp(-inf) and factor stay 0
            const float ms = mn == -INFINITY ? 0.0f : mn;
            const float corr = exp_neg_fast(m[g] - ms);
            m[g] = mn;
            float psum = 0.0f;
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float pr = exp_neg_fast(S[g][b][r] - ms);
                    psum += pr;
                    const float ps = pr * kPaPScale;
                    const _Float16 hi = (_Float16)ps;
                    P[g][b][r] = lo_col ? (_Float16)(ps - (float)hi) : hi;
                }
            lsum[g] = fmaf(lsum[g], corr, psum);
            // O's rows 4 lg + r are slots (4 lg + r) & 7, whose factor sits in
            // lane slot of lane group 0
            float cr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float c_lo = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(corr), r));
                const float c_hi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(corr), 4 + r));
                cr[r] = (lg & 1) ? c_hi : c_lo;
            }
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) O[g][n][r] *= cr[r];
        }
        // O += P' V: B fragments through transposing LDS reads (as the decode
        // kernel's), each shared by the two row groups
        auto vfrag = [&](int b, int n) {
            const int vr = 16 * b + 4 * lg + (col >> 2);
            const uint8_t* vrow = vst + vr * PITCH + 8 * (col & 1);
            const int p = (2 * n + ((col & 3) >> 1)) ^ (2 * (vr & 3));
            return __builtin_bit_cast(pa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                 (pa_lds_tr4*)(vrow + 16 * p)));
        };
#pragma unroll
        for (int bp = 0; bp < 2; ++bp)
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const pa_h8 v = pa_cat(vfrag(2 * bp, n), vfrag(2 * bp + 1, n));
#pragma unroll
                for (int g = 0; g < 2; ++g)
                    O[g][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        pa_cat(P[g][2 * bp], P[g][2 * bp + 1]), v, O[g][n], 0, 0, 0);
            }
    }

    // hi + lo rows (lane groups 2, 3 hold the lo rows of groups 0, 1), the
    // column's probability sum, and the outputs
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        float l = lsum[g];
        l += __shfl_xor(l, 16, kWave);
        l = xor32_sum(l);
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) O[g][n][r] = xor32_sum(O[g][n][r]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int s = 4 * (lg & 1) + r;  // the slot of row r
            const float den = __shfl(l, s, kWave);
            const bool empty = __shfl(lim[g], s, kWave) == 0;
            const bool nan = __shfl((int)poison[g], s, kWave);
            int tok, head;
            row_of(g, s, tok, head);
            if constexpr (SPLIT) {
                const int len = __shfl(lim[g], s, kWave);
                const float mx = __shfl(m[g], s, kWave);
                if (len > chunk) {  // (its later chunks that hold positions, and the first)
                    if (lg < 2 && tok < T && c0 < len) {
                        float* rec = ws + (((int64_t)tok * n_heads + head) * gridDim.z + blockIdx.z) *
                                              (HD + 2);
#pragma unroll
                        for (int n = 0; n < NB; ++n)
                            rec[16 * n + col] = nan ? NAN : O[g][n][r] * (1.0f / kPaPScale);
                        if (col == 0) {
                            rec[HD] = mx;
                            rec[HD + 1] = den;
                        }
                    }
                    continue;
                }
                if (c0 > 0) continue;
            }
            if (lg < 2 && tok < T) {
                float* o = out + (int64_t)tok * ld_out + (int64_t)head * HD + col;
#pragma unroll
                for (int n = 0; n < NB; ++n)
                    o[16 * n] = empty ? 0.0f : nan ? NAN : O[g][n][r] * (1.0f / kPaPScale) / den;
            }
        }
    }
}

template <int HD>
int pa_launch(float* out, int64_t ld_out, const float* q, int64_t ld_q, const void* k,
              const void* v, int64_t ld_pos, const int32_t* lens, int T, int n_ctx, int n_heads,
              int group, float scale, float* ws, size_t ws_bytes, hipStream_t stream) {
    const int G = group % 8 == 0 ? 8 : group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const int TQ = kPaRows / G, tiles = (T + TQ - 1) / TQ;
    // As many chunks as leave kPaTarget workgroups, of kPaChunkMin positions
    // or more, and as their records fit in ws.
    int64_t nch = kPaTarget / ((int64_t)tiles * (n_heads / G));
    const int64_t fit = (int64_t)(ws_bytes / ((size_t)T * n_heads * (HD + 2) * sizeof(float)));
    if (nch > fit) nch = fit;
    if (nch > n_ctx / kPaChunkMin) nch = n_ctx / kPaChunkMin;
    int chunk = n_ctx;
    if (nch > 1) {
        chunk = (int)((n_ctx + nch - 1) / nch + kPaTile - 1) / kPaTile * kPaTile;
        nch = (n_ctx + chunk - 1) / chunk;
    }
    const bool split = nch > 1;
    auto* kern = split ? pf_attention_kernel<HD, true> : pf_attention_kernel<HD, false>;
    const int rc = launch(kern, dim3((unsigned)tiles, (unsigned)(n_heads / G), split ? (unsigned)nch : 1u),
                          dim3(256), 2 * 2 * kPaTile * HD * 2, stream, lens, T, n_ctx, G, group,
                          static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), ld_pos, q,
                          ld_q, scale, out, ld_out, chunk, n_heads, ws);
    if (rc != JINF_HIP_OK || !split) return rc;
    return attn_combine_launch(out, ld_out, ws, lens, n_ctx, T, n_heads, HD, (int)nch, chunk, stream);
}

}  // namespace

int pf_attention(float* out, int64_t ld_out, const float* q, int64_t ld_q, const void* k,
                 const void* v, int kv_type, int64_t ld_pos, const int32_t* lens, int T,
                 int n_ctx, int head_dim, int n_heads, int n_heads_kv, float* ws, size_t ws_bytes,
                 hipStream_t stream, bool* launched) {
    *launched = false;
    // buffer offsets are 32 bits, reads and q rows 16-byte aligned
    if (kv_type != JINF_HIP_F16 || (head_dim != 64 && head_dim != 128) || !aligned(k, 16) ||
        !aligned(v, 16) || !aligned(q, 16) || ld_pos % 8 != 0 || ld_q % 4 != 0 ||
        (int64_t)n_ctx * ld_pos * 2 > 0x7FFFFFFF || n_heads > 65535 || T <= 0)
        return JINF_HIP_OK;
    const float scale = (float)(1.0 / sqrt((double)head_dim));
    const int group = n_heads / n_heads_kv;
    const int rc = head_dim == 64
                       ? pa_launch<64>(out, ld_out, q, ld_q, k, v, ld_pos, lens, T, n_ctx, n_heads,
                                       group, scale, ws, ws_bytes, stream)
                       : pa_launch<128>(out, ld_out, q, ld_q, k, v, ld_pos, lens, T, n_ctx, n_heads,
                                        group, scale, ws, ws_bytes, stream);
    *launched = rc == JINF_HIP_OK;
    return rc;
}

}  // namespace jinf
