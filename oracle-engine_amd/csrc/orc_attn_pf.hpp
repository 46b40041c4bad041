// Prefill attention over the library's workspace (orc_attn_pf.hip), called by
// orc_attn_prefill (orc_ops.hip).
#pragma once
#include "orc_internal.hpp"

namespace orc {

struct FaArgs {
    const float* qkv;
    int ldqkv, n_tok, n_heads, n_kv, start;
    const float2* rope;
    float *kc, *vc;
    int ctx;
    float* out;
    int ldo;
    hipStream_t s;
};

// Workspace bytes of the split K and V of p_end positions.
size_t fa_bytes(int head_dim, int n_kv, int p_end);
// The launches (head_dim 64 or 128, at most 8 query heads per kv head) on the
// workspace, between pf_ws_begin and pf_ws_end.
int fa_launch(int head_dim, const FaArgs& a, uint8_t* work, hipEvent_t start, hipEvent_t stop);

}  // namespace orc
