// Entry points shared between the C ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "awa_plan.h"
#include "seedvr2_awa.h"

namespace awa
{

// Sets the calling thread's awa_last_error() text.
void set_error(const std::string& message);

// Caller-provided device memory for the per-window text rows.
struct Scratch
{
    void* ptr;
    size_t bytes;
};

// awa_forward (norm null) or awa_forward_qknorm, with an optional event
// recorded between the attention kernel and the text-mean kernel (for
// per-kernel timing). scratch null: the text rows go to the plan's
// workspace (allocated on first use, with the work list). scratch set: they
// go there, and nothing is allocated; the plan must already hold the work
// list for the head count.
int forward_fused(const awa_plan* plan, const awa_blob* video_qkv, const awa_blob* text_qkv, const awa_qk_norm* norm,
                  const awa_blob* video_out, const awa_blob* text_out, int compute, hipStream_t stream,
                  hipEvent_t after_attention, const Scratch* scratch = nullptr);

// Resolves the current device's address of awa_forward_noalloc's static
// scratch array (once per device); AWA_ERR_DEVICE with the reason set if the
// runtime cannot.
int noalloc_setup();

} // namespace awa

// One GEMM step of the DiT block (csrc/dit_gemm.hip) on device operands, with
// the tile shape given (tests; tile < 0: the estimate's, returned in tile).
// rows[1] = 0: no text problem. Rows are contiguous; split makes the fp16 planes
// in memory of its own and waits for the stream.
struct awa_gemm_step
{
    int split, tile, epilogue, n, k;
    int rows[2], twice[2];
    const void *a[2], *w[2], *w2[2], *residual[2];
    const float *bias[2], *gate[2];
    void* out[2];
};

extern "C" int awa_gemm_step_run(awa_gemm_step* step, void* stream);

// The estimate's tile shape for a step (no device is touched).
extern "C" int awa_gemm_step_tile(const awa_gemm_step* step);

// Whether awa_dit_block_forward runs the block's GEMMs on the library (tests).
extern "C" int awa_dit_block_on_library(const awa_dit_block* block, const awa_dit_branch_weights* video_weights,
                                        const awa_dit_branch_weights* text_weights);
