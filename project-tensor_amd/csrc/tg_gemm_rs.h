// Internal entry of the register-staged GEMM (tg_gemm_rs.hip).
#pragma once
#include "tg_common.h"

// How an fp32 product runs: the kernel (see tg_gemm_rs.hip), and the K split: batch entry
// s of S multiplies k in [s*kc, min(K, (s+1)*kc)).
struct TgRsPlan {
  int shape;
  int64_t S, kc;
};

// Whether fp32 products of this size run here: all but those below 2^28 multiply-adds
// with no extent past 2048, which stay on tg_gemm.hip's fp32 kernels.  Those are bound by
// launch and memory latency (32x256x784: 20 us there, 15 us here; 512^3: 19 and 17 us),
// and an MLP's products are among them, whose sums keep their order: Adam's first steps
// divide a gradient by its own magnitude, so a gradient that cancels to rounding level
// turns another order of the same sum into a visibly different weight.
inline bool tg_gemm_rs_serves(int64_t M, int64_t N, int64_t K, int64_t batch) {
  return M > 2048 || N > 2048 || K > 2048 ||
         (double)M * (double)N * (double)K * (double)batch >= 268435456.0;
}

// The fastest of the kernels for `batch` products of M x N x K, K split only where
// can_split.  tn: A transposed, B plain.
TgRsPlan tg_gemm_rs_plan(bool tn, int64_t M, int64_t N, int64_t K, int64_t batch,
                         bool can_split);

// C[z] = alpha * op(A[z]) @ op(B[z]) + beta * C[z] (+ bias) in fp32, any extents, leading
// dimensions and alignment (element alignment is enough).  Without a split (p.S = 1) z
// is the batch entry; with one, batch is p.S, the strides are those of a chunk of kc and
// K is the whole extent.
int tg_gemm_rs(const TgRsPlan& p, int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha,
               const float* A, int64_t lda, int64_t sa, const float* B, int64_t ldb, int64_t sb,
               float beta, float* C, int64_t ldc, int64_t sc, int64_t batch, const float* bias,
               hipStream_t s);
