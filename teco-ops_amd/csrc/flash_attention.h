// flash_attention.h — host-side types of the flash-attention entry points,
// shared by flash_attention.hip (kernels, planning, the C entry points) and
// fa_noalloc.hip (the allocation-free entry point and its static scratch).
#pragma once

#include <cstddef>
#include <cstdint>

#include "common.h"

namespace tecoops {
namespace fa {

// Kernel parameters (passed by value to every flash-attention kernel).
struct FaParams {
    const uint16_t *q;
    const uint16_t *kc;
    const uint16_t *vc;
    uint16_t *o;
    const int *bt;
    long long bt_stride;
    const int *q_lens;   // per-sequence q lengths, or NULL
    const int *cu_q;     // cumulative q offsets [batch+1], used when q_lens is NULL
    const int *kv_lens;
    int batch, H, Hkv, G, bs, lbs, num_blocks;  // lbs = log2(bs) when bs is a power of 2
    int kv_cap;          // block-table width * block_size: kv lengths are clamped to it
    long long page_stride;                      // Hkv * bs * D elements per cache block
    float scale_log2;    // softmax_scale * log2(e)
    float inv_scale_log2;  // 1 / scale_log2: the rescale test compares raw scores
    int causal;
    int turn;            // grid rows after which the sequences' places move on, as a shift
    long long total_q;   // rows of q and of the output (q's descriptor)
    // split-KV decode
    float *ws_o;         // [B][Hkv][max_splits][ncols][D]
    float *ws_ml;        // [B][Hkv][max_splits][ncols][2]
    int split_len, max_splits, rq, ncols;
    bool direct;         // decode workgroups take their item in grid order
    void *ws_plan;       // split prefill: the plan (the states are in ws_o)
};

// Launch shape.  rq is the host's bound on q_len (routing and grid height),
// rk its bound on kv_len (prefill routing), split_len / max_splits the
// split-KV plan from rk.  Neither bound changes the output (the kernels also
// cover longer sequences), only the speed.
struct Plan {
    bool decode;
    int rq, rk, ncols, split_len, max_splits;
};

// Prefill over split keys (fa_split.hip): `slots` pieces share the batch's
// work, none shorter than `least` keys; wide selects the 12-wave kernels.
// slots 0: not split.
struct SplitArgs {
    int slots, least, wide;
};
constexpr int kSplitMaxBatch = 64;        // sequences of a split prefill
constexpr size_t kSplitPlanBytes = 2048;  // the workspace starts with the plan

// A validated call: kernel parameters, launch shape and element type.
struct FaCall {
    FaParams p;
    Plan pl;
    SplitArgs split;  // the split prefill the call may take, given a workspace
    int D;
    bool bf16;
};

// Argument checks of reference flash_attention.cpp:44-69 and the launch plan
// (fixed_hints: the hints as given, for a workspace sized from them).
tecoopsStatus_t prepare(tecoopsHandle_t handle, int max_seqlen_q, int max_seqlen_k,
                        const int *q_seq_lens, const int *cu_seqlens_q, const int *kv_seq_lens,
                        const tecoopsTensorDescriptor_t btDesc, const void *blockTable,
                        const tecoopsTensorDescriptor_t qDesc, const void *qData,
                        const tecoopsTensorDescriptor_t kDesc, const void *kCache,
                        const tecoopsTensorDescriptor_t vDesc, const void *vCache,
                        const tecoopsTensorDescriptor_t oDesc, void *oData, float softmax_scale,
                        int causal, bool fixed_hints, FaCall &c);

// Bytes of split-KV partials the call needs (0 for prefill).
size_t workspace_bytes(const FaCall &c);

// The same from the sizes alone (H a multiple of Hkv), for a workspace of this
// call's kv heads where tecoopsGetFlashAttentionWorkspaceSize covers any number.
size_t workspace_bytes(int batch, int H, int Hkv, int D, int q_hint, int k_hint);

// Bytes of partial states of a split prefill, and its launch (p.ws_o holds
// them).
size_t split_bytes(const SplitArgs &a, int D);
tecoopsStatus_t launch_split(hipStream_t s, const FaParams &p, const SplitArgs &a, int D, bool bf16);

// Enqueues the call on stream s, its split-KV partials in ws.
tecoopsStatus_t launch(hipStream_t s, FaCall &c, void *ws);

}  // namespace fa
}  // namespace tecoops
