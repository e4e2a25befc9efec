/* C ABI of the gfx950 plain bf16 products (same library and conventions as
 * mm1_attn.h: bf16 tensors as `void*`, the HIP stream as `void*`, caller-owned
 * buffers, no allocation, no synchronisation, return 0 / a negative MM1_E_*
 * code / a positive hipError_t).
 *
 * The products around the SwiGLU and cross-entropy kernels and the
 * projections' weight gradients, which the reference runs as torch GEMMs
 * (swiglu_tilelang.py:284-301, lm_head_tilelang.py:226-243,
 * attention_tilelang.py:470-472 and :518).
 */
#ifndef MM1_GEMM_H
#define MM1_GEMM_H

#include <stddef.h>

#include "mm1_attn.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Layout of an operand: MM1_GEMM_ROW has the reduction index contiguous
 * (x [M, K], w [N, K]), MM1_GEMM_COL has it outermost (x [K, M], w [K, N]). */
#define MM1_GEMM_ROW 0
#define MM1_GEMM_COL 1

/* Bytes of scratch mm1_gemm needs for this shape in any layouts, with (joined)
 * or without a w1 (0 for many): fp32 partial sums where K is split over several
 * workgroups. */
size_t mm1_gemm_workspace_size(int M, int N, int K, int joined);

/* Modelled time of mm1_gemm at this shape on the current device, in us
 * (negative for sizes it refuses). */
double mm1_gemm_estimate_us(int M, int N, int K);

/* out[m][n] = sum_k x(m, k) w(n, k): bf16 operands, fp32 accumulation over
 * all of K, rounded once to bf16 (out_f32 = 0) or stored in fp32 (1).
 * ldx, ldw, ldo: row strides in elements.
 *   w1, k_cut: with w1 != NULL, w holds k < k_cut and w1 (same layout and
 *     stride) the rest; k_cut a multiple of 64.  Else k_cut = 0.
 *   out1, n_cut: with out1 != NULL, out holds the columns below n_cut and out1
 *     (same stride) the others; n_cut a multiple of 64.  Else n_cut = 0.
 * x ROW with w ROW or COL, or both COL (MM1_E_SHAPE for x COL with w ROW).
 * M, N, K >= 1, K a multiple of 128 unless both are COL (then any K, at most
 * 2^28), N a multiple of 8 (and M when x is COL),
 * every stride a multiple of 8 and at least its row's length, 16-byte aligned
 * pointers; the bytes of 256 rows of a ROW operand and of 64 rows of a COL
 * operand below 2^31, M and N at most 2^28, at most 2^24 output tiles of
 * 256 x 256.  Deterministic. */
int mm1_gemm(const void* x, int x_layout, long ldx, const void* w, int w_layout, long ldw, const void* w1,
             int k_cut, void* out, void* out1, int n_cut, long ldo, int out_f32, void* workspace,
             size_t workspace_bytes, int M, int N, int K, void* stream);

/* dst = the fp32 tensors src0 .. src3 rounded to bf16 (nearest even), one
 * after the other (n0 .. n3 values, each a multiple of 8, 0 for none): the
 * operands of a product whose activations and weights are held in fp32. */
int mm1_cast_bf16(const float* src0, long n0, const float* src1, long n1, const float* src2, long n2,
                  const float* src3, long n3, void* dst, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* MM1_GEMM_H */
