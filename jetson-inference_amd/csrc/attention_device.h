// Device code shared by the fp16-cache (attention.hip) and fp32-cache
// (attention_f32.hip) decode attention: the merge of a context split over
// several workgroups, whose records {O[HD], m, l} per (sequence, head, chunk)
// both kernels write alike.
#pragma once

#include "jinf_device.h"

namespace jinf {

// Below kAmInKernelMerge (sequence, head group) pairs a split context is
// merged by the attention kernel itself, at or above it by a second launch.
// The merge's counters, one per pair, are 16-bit counts, two to a word, in
// the first kAmCounterBytes of the workspace whatever the call's shape, and
// every call's records start at or past them.  So calls of any shapes share a
// workspace: none writes records where another one keeps its counters.
constexpr int kAmInKernelMerge = 128;
constexpr size_t kAmCounterBytes = kAmInKernelMerge * sizeof(uint16_t);

// Reference point of a row's exponentials: its largest score, or 0 when it
// has none above -inf (then exp(-inf - 0) = 0, not NaN).  Maxima skip NaN
// scores, so a row with one keeps it in its probability sum and outputs,
// which stay NaN through every merge whatever the row's maximum is.
__device__ __forceinline__ float softmax_ref(float m) { return m > -INFINITY ? m : 0.0f; }

// The in-kernel merge of a split context (the kernels' MERGE form): the
// calling workgroup has stored its records for head slots [h0, h0 + G) of
// sequence s.  `lds` is the kernel's dynamic LDS, free at this point.
template <int HD>
__device__ __forceinline__ void am_merge_last(float* __restrict__ out, int64_t ld_out,
                                              float* __restrict__ ws,
                                              unsigned* __restrict__ counters, int s, int n_heads,
                                              int h0, int G, int nch, int used, uint8_t* lds) {
    constexpr int MS = HD + 2;
    // The last of the `used` workgroups of this (sequence, head group) merges
    // their records in chunk order and returns the counter to zero.  Records
    // are written and read with device-coherent accesses (they bypass the
    // per-XCD L2 caches, which are not coherent with one another).  Ordering:
    // every thread waits for its record stores, the barrier (a workgroup-scope
    // release / acquire) orders them before thread 0's counter update, an
    // agent-scope release increment; the workgroup that sees the final count
    // then acquires, so it synchronizes with every earlier release, and its
    // threads read the records after the barrier that follows.  Only the
    // merging workgroup pays the acquire's L2 invalidation.  (Agent-scope
    // release fences in every wave instead cost 19 -> 28 us at batch 1, 8192
    // positions: each writes back the whole L2.  A relaxed increment, relying
    // on the device-coherent accesses alone, measured the same as this on the
    // decode and 70B attention workloads.)
    __shared__ int am_last;
    __builtin_amdgcn_s_waitcnt(waitcnt_vm<0>());
    __syncthreads();
    if (threadIdx.x == 0) {
        // (a count stays below 2048: the merge's LDS bounds the chunks)
        const unsigned i = s * gridDim.x + blockIdx.x, shift = 16 * (i & 1);
        unsigned* cnt = counters + (i >> 1);
        const unsigned prev =
            __hip_atomic_fetch_add(cnt, 1u << shift, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        am_last = ((prev >> shift) & 0xFFFFu) + 1 == (unsigned)used;
        if (am_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (am_last)
            __hip_atomic_fetch_sub(cnt, (unsigned)used << shift, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!am_last) return;
    // Merge: the chunks' (m, l) pairs and weights f_c = exp(m_c - M) go
    // through LDS (the tile buffers are free now), computed once per (chunk,
    // head) in parallel; then each (head, dim) sums f_c O_c[d] over the chunks
    // with the loads of several chunks in flight.  Same operations in the same
    // order per output as a sequential merge.
    float* mw = reinterpret_cast<float*>(lds);  // [used][8]: m, then f
    float* ml = mw + used * 8;                  // [used][8]: l
    float* mM = ml + used * 8;                  // [8]: reference point per head slot
    for (int idx = threadIdx.x; idx < used * G; idx += blockDim.x) {
        const int c = idx / G, g = idx % G;
        const float* e = ws + (((int64_t)s * n_heads + h0 + g) * nch + c) * MS;
        mw[c * 8 + g] = rec_load(e + HD);
        ml[c * 8 + g] = rec_load(e + HD + 1);
    }
    __syncthreads();
    if (threadIdx.x < G) {
        float M = -INFINITY;
        for (int c = 0; c < used; ++c) M = fmaxf(M, mw[c * 8 + threadIdx.x]);
        mM[threadIdx.x] = softmax_ref(M);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < used * G; idx += blockDim.x) {
        const int c = idx / G, g = idx % G;
        mw[c * 8 + g] = exp_neg_fast(mw[c * 8 + g] - mM[g]);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * HD; idx += blockDim.x) {
        const int g = idx / HD, d = idx % HD;
        const float* rec = ws + ((int64_t)s * n_heads + h0 + g) * nch * MS + d;
        float num = 0.0f, den = 0.0f;
#pragma unroll 8
        for (int c = 0; c < used; ++c) {
            const float f = mw[c * 8 + g];
            num = fmaf(f, rec_load(rec + (int64_t)c * MS), num);
            den = fmaf(f, ml[c * 8 + g], den);
        }
        out[(int64_t)s * ld_out + (int64_t)(h0 + g) * HD + d] = num / den;
    }
}

// Merges the chunk records [sequence][head][nch] of every row whose context
// does not fit in one chunk (attn_combine_kernel).
int attn_combine_launch(float* out, int64_t ld_out, const float* ws, const int32_t* lens,
                        int n_past, int n_seq, int n_heads, int head_dim, int nch, int chunk,
                        hipStream_t stream);

// The fp32-cache kernel (attention_f32.hip): G query heads of a kv head per
// workgroup, chunks of `chunk` positions; counters null: split contexts are
// left to attn_combine_kernel.
int attn_f32_launch(float* out, int64_t ld_out, const float* q, int64_t ld_q, const void* k,
                    const void* v, int64_t ld_pos, int64_t ld_seq, const int32_t* lens,
                    int n_past, int n_seq, int head_dim, int n_heads, int group, int G, int chunk,
                    int nch, float scale, float* ws, unsigned* counters, hipStream_t stream);

}  // namespace jinf
