// Internal entry of the few-row MFMA matmul (skinny.hip), used by the decode launchers.
#pragma once

#include <hip/hip_runtime.h>

#include "qmm_blocks.h"

// From this many activation rows on, Q4_K and Q6_K weights of k columns go through the MFMA few-row kernel, which decodes
// each weight block once for all rows.  Measured on MI355X, the matvec against it: three rows Q4_K 14336x4096 12.6 and
// 9.9 us, 4096x4096 5.7 and 5.0, Q6_K 1024x4096 7.4 and 5.3; two rows 14336x4096 10.5 and 9.9 but 4096x4096 4.7 and 5.0,
// Q6_K 1024x4096 3.1 and 5.3; two rows of wide weights Q6_K 4096x14336 17.9 and 14.4, Q4_K 8192x8192 14.3 and 11.1.
inline int qmm_skinny_min_rows(int64_t k) { return k >= 8192 ? 2 : 3; }

// The same for Q8_0 / Q4_0 / Q5_0 and Q5_K weights of n rows.  The kernel's time does not grow with the rows, the matvec's
// does; narrow weights leave the kernel with few workgroups.  MI355X, us, matvec and this kernel, Q8_0 unless said
// otherwise: 1024x4096 8 rows 5.2 / 5.6, 16 rows 9.8 / 5.6; 2048x4096 5 rows 5.6 / 6.0, 6 rows 6.5 / 6.0; 4096x4096 3 rows
// 7.0 / 7.3, 4 rows 8.3 / 7.3; 4096x14336 3 rows 21.8 / 15.5; 14336x4096 3 rows 16.5 / 14.2, 16 rows 60.6 / 14.7, Q5_K 3
// rows 13.8 / 12.7, Q4_0 12.1 / 10.2, Q5_0 13.3 / 12.3; 2 rows 14.0 / 14.9.
inline int qmm_skinny_b32_min_rows(int64_t n, int64_t k) {
  return n < 2048 ? 9 : n < 4096 ? 6 : n < 8192 && k < 8192 ? 4 : 3;
}
// Fused forms of the 32-value types.  Gate and up, 2 x n rows: 2 x 2048x2048 4 rows 5.7 / 5.6, 6 rows 9.8 / 5.6; 2 x
// 14336x4096 2 rows 23.0 / 23.8, 3 rows 29.7 / 23.6, 16 rows 115 / 25.  Q, K and V are three launches here and one matvec:
// (2048 + 2 x 512)x2048 6 rows 10.4 / 12.0, 8 rows 11.9 / 11.9; (4096 + 2 x 1024)x4096 4 rows 14.4 / 18.6, 8 rows 26.9 /
// 18.7.
inline int qmm_skinny_b32_min_rows_glu(int64_t n) { return n < 4096 ? 5 : 3; }
constexpr int QMM_SKINNY_B32_MIN_ROWS_QKV = 8;

// Decode-layout activations (b rows of Q8_K blocks, stride_col_y blocks apart) against Q4_K / Q5_K / Q6_K weights;
// dst[j * stride_col_dst + row] of element type out_type (QMM_TYPE_F32 / F16 / BF16).  Returns false, launching
// nothing, for a case it does not serve (other weight types, b outside 1..32 (Q5_K 1..16),
// K not a multiple of 256).
bool qmm_skinny_decode(int type, int out_type, const void *vx, const void *vy, void *dst, int ncols_x, int nrows_x,
                       int stride_col_y, int stride_col_dst, int b, hipStream_t s);

// The same for the fused GLU form: dst[j * stride_col_dst + row] = act(W_gate . y_j) * (W_up . y_j).
bool qmm_skinny_glu(int type, int out_type, const void *vx_gate, const void *vx_up, const void *vy, void *dst,
                    int ncols_x, int nrows_x, int stride_col_y, int stride_col_dst, int b, int activation,
                    hipStream_t s);

// The same for Q8_0 / Q4_0 / Q5_0 weights against rows of Q8_0 blocks (stride_col_y blocks apart), b in 1..16; vx2: the
// up weights of the GLU form, null for a plain product.
bool qmm_skinny_b32(int type, int out_type, const void *vx, const void *vx2, const void *vy, void *dst, int ncols_x,
                    int nrows_x, int stride_col_y, int stride_col_dst, int b, int activation, hipStream_t s);

// The same over the tensor-core entries' activation layout (rows of ncols_x / 256 blocks {f32 d; int8 qs[256]},
// units.h), for launch_mmvq_tc_gguf_<t>_*_plain.
bool qmm_skinny_tc(int type, int out_type, const void *vx, const void *vy, void *dst, int ncols_x, int nrows_x,
                   int stride_col_dst, int b, hipStream_t s);

// Expert-grouped matmul (launch_mmq_gguf_<t>_moe) over prefill-layout activations when the experts receive few rows each:
// at most QMM_SKINNY_MOE_ROWS on average.  dst[ids_dst[m] * ldd + n], f32.  Returns false, launching nothing, for a case
// it does not serve.  The whole step of 8 x Q4_K experts of 14336x4096 / 4096x14336, top-2, MI355X, against the grouped
// tile kernel: 4 rows an expert on average 167 and 249 us, 16 rows 219 and 250, 32 rows 289 and 327, 64 rows 454 and 441.
#ifndef QMM_SKINNY_MOE_ROWS
#define QMM_SKINNY_MOE_ROWS 32
#endif
bool qmm_skinny_moe(int type, const void *x, const void *y, const int32_t *ids_dst, const int32_t *bounds, float *dst,
                    int64_t ncols_x, int64_t nrows_x, int64_t w_row_bytes, int64_t ncols_dst, int64_t ldd,
                    int64_t num_experts, hipStream_t s);

// The same for gate and up in one launch: dst[m * ldd + n] = act(W_gate . y_m) * (W_up . y_m), row m of the activations.
bool qmm_skinny_moe_glu(int type, const void *gate, const void *up, const void *y, const int32_t *bounds, float *dst,
                        int64_t ncols_x, int64_t nrows_x, int64_t w_row_bytes, int64_t ncols_dst, int64_t ldd,
                        int64_t num_experts, int activation, hipStream_t s);
