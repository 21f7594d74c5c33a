// A library with the entry points that the native operator calls bind to. Its add waits, at most ten seconds, until
// open_gate() is called: a caller that keeps every other Python thread from running meanwhile gets an error.
#include <atomic>
#include <chrono>
#include <thread>

#define API extern "C" __attribute__((visibility("default")))
#define REFUSES(name) API int name() { return -1; }

static std::atomic<bool> gate{false};
API void open_gate() { gate = true; }
API int mi_add_inplace() {
    for (int i = 0; i < 1000 && !gate; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    return gate ? 0 : -1;
}
API const char* mi_last_error() { return "the gate stayed closed"; }
API unsigned long mi_sdpa_split_scratch_bytes() { return 0; }
API unsigned long mi_attn_block_scratch_bytes() { return 0; }
API unsigned long mi_linear_attn_workspace_bytes() { return 0; }
API unsigned long mi_linear_attn_scratch_bytes() { return 0; }
REFUSES(mi_sdpa_forward)
REFUSES(mi_rope_apply)
REFUSES(mi_headnorm_rope)
REFUSES(mi_linear_forward)
REFUSES(mi_linear_forward_n)
REFUSES(mi_linear_geglu_forward)
REFUSES(mi_rms_norm_forward)
REFUSES(mi_rms_norm_pair_forward)
REFUSES(mi_flash_attention_qkvo_forward)
REFUSES(mi_flash_attention_q_with_kv_cached_forward)
REFUSES(mi_linear_attn_relu_forward)
