// Internal interface of the prompt path (prefill.hip) for the batch decoder:
// one layer's matrix products over many tokens of one prompt at once.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace jinf {

// Prompt tokens per step of the wide path, and per workgroup of its matrix
// products (buffers are padded to a multiple of the latter).
constexpr int kPfMaxRows = 1024;
constexpr int kPfTile = 128;

// The wide path's device buffers, carved out of one allocation.
struct PfBuf {
    int rows = 0;            // tokens they hold (a multiple of kPfTile)
    uint8_t* rec = nullptr;  // x as matrix-core fragments
    float* xs = nullptr;     // the prepared x's scales: [128-token tile][slab][1 / s, s][128]
    float2* cs = nullptr;    // [rows][head_dim / 2] RoPE cos, sin
    float* part = nullptr;   // partial sums of split columns
    size_t part_bytes = 0;
};

// A residual add left pending: k partial sums [k][rows][cols], merged into h
// by the next pf_prepare of h (k 0: nothing pending).
struct PfPend {
    int k = 0;
};

// Bytes of the buffers for `rows` tokens of a model (part included).
size_t pf_rec_bytes(int rows, int cols);
size_t pf_part_bytes();

// RoPE table of positions[0 .. T).
int pf_rope_table(const PfBuf& b, const int32_t* positions, int T, int head_dim, float freq_base,
                  hipStream_t stream);

// x [T][cols] (h with a pending residual add merged and written back first)
// into b.rec, RMS-normalised when norm_w is given.
int pf_prepare(const PfBuf& b, float* x, int ld_x, int T, int cols, const void* norm_w,
               int norm_type, float eps, PfPend* pend, hipStream_t stream);

// Completes a pending residual add into x (nothing without one).
int pf_merge(const PfBuf& b, float* x, int ld_x, int T, int cols, PfPend* pend,
             hipStream_t stream);

// y[t] (+)= W x[t] from the prepared x; accum with split columns leaves the
// add pending (*pend).
int pf_matmul(const PfBuf& b, const void* w, int qtype, int T, int rows, int cols, float* y,
              int ld_y, bool accum, PfPend* pend, hipStream_t stream);

// y[t][i] = silu(W_gate x[t])_i (W_up x[t])_i.
int pf_swiglu(const PfBuf& b, const void* w_gate, const void* w_up, int qtype, int T, int n_ff,
              int cols, float* y, int ld_y, hipStream_t stream);

// Q / K / V (matrices of one format; null ones skipped) with RoPE from the
// table and the cache rows at positions[t].
int pf_qkv(const PfBuf& b, const void* wq, const void* wk, const void* wv, int qtype, int T,
           int cols, float* q, int ld_q, void* kc, void* vc, int kv_type,
           const int32_t* positions, int max_ctx, int head_dim, int n_heads, int n_heads_kv,
           hipStream_t stream);

// Attention of T rows of one sequence over its cache (k, v: its position 0;
// at most n_ctx positions), row t over positions below lens[t].  ws: scratch
// for the records of split contexts, any contents.  *launched false (status
// 0, nothing enqueued): a cache type, head size or alignment it does not take.
int pf_attention(float* out, int64_t ld_out, const float* q, int64_t ld_q, const void* k,
                 const void* v, int kv_type, int64_t ld_pos, const int32_t* lens, int T,
                 int n_ctx, int head_dim, int n_heads, int n_heads_kv, float* ws, size_t ws_bytes,
                 hipStream_t stream, bool* launched);

}  // namespace jinf
