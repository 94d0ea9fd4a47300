// gemm_x3.h — the FP32 product on bf16 MFMA (gemm_x3.hip), chosen by cf_gemm_plan.
#ifndef CF_GEMM_X3_H_
#define CF_GEMM_X3_H_

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "kernels.h"

// The DMA kernels step their W (K, N) addresses by a stage of rows in 32 bits (64 fp16 rows,
// 32 fp32 ones): every segment narrower than 2^25 columns.  Wider ones take the
// register-staged kernels, which index in 64 bits.
inline bool gemm_w_steps_fit(const cf_gemm_args_t* a) {
    for (int s = 0; s < a->nseg; s++)
        if (!a->w_nk && a->n[s] >= 1 << 25) return false;
    return true;
}

// The tile for this product (an index for gemm_x3_launch), or -1 where it does not apply.
// *ks: the ranges of k its workgroups sum; *clk: its estimated time in CU clocks.
int gemm_x3_pick(const cf_gemm_args_t* a, int* ks, float* clk);
// Workspace floats (a->partials) of a launch with a->ksplit ranges.
size_t gemm_x3_floats(const cf_gemm_args_t* a);
int gemm_x3_launch(const cf_gemm_args_t* a, int pick, hipStream_t st);
// FP32 products of few rows on the fp32 MFMA (gemm_f32_ws.hip), likewise.
int gemm_f32_ws_pick(const cf_gemm_args_t* a, int* ks, float* clk);
size_t gemm_f32_ws_floats(const cf_gemm_args_t* a);
int gemm_f32_ws_launch(const cf_gemm_args_t* a, int pick, hipStream_t st);
// FP16 products whose operands are FP32 in memory (a->mix), with a->ksplit ranges of k.
int32_t gemm_mix_ok(const cf_gemm_args_t* a);
int gemm_mix_launch(const cf_gemm_args_t* a, hipStream_t st);
// Sums a->ksplit ranges of fp32 partial sums at a->partials into out[0] (gemm.hip).
int gemm_splitk_sum_launch(const cf_gemm_args_t* a, hipStream_t st);

#endif  // CF_GEMM_X3_H_
