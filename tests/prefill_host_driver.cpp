// The prompt path's host side without a GPU: this program defines the HIP
// calls that the library makes (device memory is host memory nobody reads,
// kernels are not run, chosen calls fail) and drives the C interface.  Prints
// one "name value" line per observation; tests/test_prefill_host.py reads them.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <vector>

#include "jinf/engine_hip.h"

static hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
static int g_strict_allocs = 0;     // allocations outside the relaxed mode
static int g_allocs = 0;
static int g_fail_sync = 0;         // the n-th stream synchronize from now fails
static int g_fail_malloc = 0;       // every device allocation fails
static std::vector<std::vector<int>> g_uploads;  // host-to-device copies

static void note_alloc() {
    ++g_allocs;
    if (g_mode != hipStreamCaptureModeRelaxed) ++g_strict_allocs;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    note_alloc();
    if (g_fail_malloc) return hipErrorOutOfMemory;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    note_alloc();
    *p = calloc(1, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void* src, size_t n, hipMemcpyKind k, hipStream_t) {
    if (k == hipMemcpyHostToDevice) {
        const int* s = static_cast<const int*>(src);
        g_uploads.emplace_back(s, s + n / 4);
    }
    return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    return g_fail_sync > 0 && --g_fail_sync == 0 ? hipErrorUnknown : hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    const hipStreamCaptureMode old = g_mode;
    g_mode = *m;
    *m = old;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
}

static void show(const char* name, int v) { printf("%s %d\n", name, v); }

int main() {
    void* w = aligned_alloc(256, 256);
    jinf_hip_layer_weights lw;
    memset(&lw, 0, sizeof lw);
    lw.attn_norm = lw.ffn_norm = w;
    lw.attn_q = lw.attn_k = lw.attn_v = lw.attn_output = w;
    lw.ffn_gate = lw.ffn_up = lw.ffn_down = w;
    lw.attn_q_type = lw.attn_k_type = lw.attn_v_type = lw.attn_output_type = 2;  // Q4_0
    lw.ffn_gate_type = lw.ffn_up_type = lw.ffn_down_type = 2;
    jinf_hip_engine_desc d;
    memset(&d, 0, sizeof d);
    d.n_layers = 1;
    d.n_embd = 256;
    d.n_heads = 4;
    d.n_heads_kv = 2;
    d.n_ff = 512;
    d.n_vocab = 300;
    d.max_context = 16;
    d.rms_norm_eps = 1e-5f;
    d.rope_freq_base = 10000.0f;
    d.kv_type = 1;
    d.token_embd = w;
    d.token_embd_type = 2;
    d.layers = &lw;
    jinf_hip_engine* e = nullptr;
    show("engine", jinf_hip_engine_create(&e, &d));
    const std::vector<int32_t> toks(1500, 7);
    for (int wide = 1; wide >= 0; --wide) {
        jinf_hip_batch* b = nullptr;
        show("batch", jinf_hip_batch_create(&b, e, 8, 2048, 1));
        show("first", jinf_hip_batch_prefill(b, 1, toks.data(), 5, nullptr));
        // a prompt of several chunks whose second chunk fails
        g_allocs = g_strict_allocs = 0;
        g_fail_malloc = !wide;
        g_fail_sync = 2;
        show("failed", jinf_hip_batch_prefill(b, 1, toks.data(), 1500, nullptr));
        g_fail_malloc = g_fail_sync = 0;
        show("allocs", g_allocs);
        show("strict_allocs", g_strict_allocs);
        show("mode_kept", g_mode == hipStreamCaptureModeGlobal);
        show("n_past", jinf_hip_batch_n_past(b, 1));
        g_uploads.clear();
        show("again", jinf_hip_batch_prefill(b, 1, toks.data(), 3, nullptr));
        show("from", g_uploads.size() > 1 && g_uploads[1].size() ? g_uploads[1][0] : -1);
        show("n_past_after", jinf_hip_batch_n_past(b, 1));
        jinf_hip_batch_destroy(b);
    }
    jinf_hip_engine_destroy(e);

    // which prompts run wide: those whose first call allocates
    const int widths[3][5] = {
        {256, 512, 4, 2, 2}, {4096, 14336, 32, 8, 2}, {4096, 14336, 32, 8, 8}};  // 8: Q8_0
    for (const auto& wd : widths) {
        d.n_embd = wd[0];
        d.n_ff = wd[1];
        d.n_heads = wd[2];
        d.n_heads_kv = wd[3];
        lw.ffn_gate_type = lw.ffn_up_type = wd[4];
        show("engine", jinf_hip_engine_create(&e, &d));
        const int calls[5][2] = {{8, 8}, {8, 9}, {8, 16}, {8, 17}, {64, 65}};
        for (const auto& c : calls) {
            jinf_hip_batch* b = nullptr;
            show("batch", jinf_hip_batch_create(&b, e, c[0], 256, 1));
            g_allocs = 0;
            show("first", jinf_hip_batch_prefill(b, 0, toks.data(), c[1], nullptr));
            show("wide", g_allocs != 0);
            jinf_hip_batch_destroy(b);
        }
        jinf_hip_engine_destroy(e);
    }
    return 0;
}
