// How attention of head_dim 512 is laid out (csrc/sdpa_wide_plan.h), for a test: pieces of the key axis, and whether the kernel for long
// calls takes the launch when `scratch` allows those pieces.
#include "sdpa_wide_plan.h"

extern "C" int wide_plan(int batch_heads, int q_len, int kv_len, int causal, int scratch, int compute_units, int* pieces) {
    mi::SdpaDev p{};
    p.B = batch_heads;
    p.H = 1;
    p.Lq = q_len;
    p.Lk = kv_len;
    p.mask_mode = causal ? MI_MASK_CAUSAL : MI_MASK_NONE;
    *pieces = scratch ? mi::sdpa::wide_split(p, 512, compute_units) : 1;
    return mi::sdpa::wide_long_pays(p, *pieces, compute_units);
}
