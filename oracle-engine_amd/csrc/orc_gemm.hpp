// Declarations shared by the two quantized GEMM translation units:
// orc_gemm.hip (vector path for Q8_0 / Q4_0, dispatch, C ABI) and
// orc_mmq.hip (matrix-core path for Q4_K / Q6_K and mixed launches).
#pragma once
#include "orc_internal.hpp"

#include <hip/hip_ext.h>

namespace orc {

// One GEMM launch: up to three weight segments sharing the activations X.
struct QmvParams {
    const uint8_t* w[3];
    float* y[3];
    const float* bias[3];
    int rows[3];
    int n_seg;
    int n_rows;  // logical rows: sum of the segment rows, or 2 x (gate, up) pairs
    int units;   // units per row
    uint64_t row_bytes;
    const float* x;
    int ldx, ldy, n_tok, n_in;
    const float* norm_w;
    float eps;
    int epi;
    int n_groups;
    int hs;               // matrix-core windowed mode: units of a wave's range staged at a time
    int seg_type[3];      // matrix-core mixed launches: weight type of each segment
    uint64_t seg_rb[3];   // and its row bytes
    int tok_block;        // tokens per token block (blockIdx.y) of a launch; n_tok counts all blocks
    int late_w;           // vector path: first weight batch issued after the activations are staged
    int split_rows;       // vector mixed launches: logical rows of the leading Q4_K segments
};

// Kernel timing of one launch: start / stop events taken from its dispatch.
struct LaunchEvents {
    hipEvent_t start = nullptr, stop = nullptr;
};

// Device properties set by gemm_device_init.
extern int g_n_cu;
extern size_t g_lds_max;

// k_mmq type parameter: Q4_K and Q6_K segments in one launch (a Q4_K_M
// layer's Q|K|V, whose attn_v is Q6_K).
constexpr int kMixK = 256;

// Matrix-core path (orc_mmq.hip): tokens per launch for this shape (0 if none
// fit), and one launch of at most that many tokens.
bool mmq_type(int type);
int mmq_max_tokens(int type, const QmvParams& p);
int mmq_launch(int type, const QmvParams& p, hipStream_t s, const LaunchEvents& ev);
// the same for launches whose wave ranges are staged in windows (orc_mmq_win.hip)
int mmq_launch_windowed(int type, const QmvParams& p, hipStream_t s, const LaunchEvents& ev);
// Captured prefill launches (orc_mmq.hip): calls of at least kPfMinTok tokens
// on one K-quant or Q8_0 type whose stream is being captured run k_mmq_pf, all
// tokens in one launch, without a workspace.
constexpr int kPfMinTok = 256;
bool mmq_prefill(int type, const QmvParams& p);
int mmq_prefill_launch(int type, const QmvParams& p, hipStream_t s, const LaunchEvents& ev);

// Prefill launches over split activations (orc_pf.hip): calls of at least
// kPfSplitMin tokens, every type but F32, whose stream is not being captured.
// The line: at 24 tokens the two launches and the split cost what the verify
// kernels' 16-token block and its remainder do on the smallest K-quant matrix
// (3072 x 3072 Q4_K: 21 us either way; at 20 tokens 21 against 18, at 32 21
// against 27); every larger or vector-kernel matrix gains earlier (7B gate+up
// Q6_K at 20 tokens 70 against 158 us). Verify passes stay below it, and small
// K-quant and dense matrices stay with the verify kernels for more tokens
// (verify_faster, orc_gemm.hip).
constexpr int kPfSplitMin = 24;
int pf_init();
void pf_release();
// The workspace of the prefill kernels (one per device): 1024 tokens of 18944
// split values (83 MB) with room for partial sums, or the split K and V of
// 32 K positions of eight 128-wide kv heads (256 MB and a word per block) with
// the partial results of 32 rows in each of 256 workgroups (4.3 MB). pf_ws_begin locks it and orders
// the stream behind its last use; kPfBusy where the caller takes a path
// without it: the stream is being captured, there is no workspace, or its last
// use was on a library stream whose capture was begun through HIP itself
// instead of orc_graph_begin. pf_ws_end ends the use and unlocks.
constexpr size_t kPfWorkBytes = (size_t)264 << 20;
constexpr int kPfBusy = 1;
int pf_ws_begin(hipStream_t s, uint8_t** buf);
int pf_ws_end(hipStream_t s);
bool pf_takes(int type, const QmvParams& p);  // the shape; pf_ws_begin says the rest
double pf_estimate(int type, const QmvParams& p);  // microseconds of a small call
int pf_launch(int type, const QmvParams& p, hipStream_t s, const LaunchEvents& ev, uint8_t* work);

}  // namespace orc
