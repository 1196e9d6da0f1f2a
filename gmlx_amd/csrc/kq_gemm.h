// Matrix-core matmul for tens to thousands of activation rows (kq_gemm.hip):
// dense groups and the dense GLU of more than 64 rows, and the MoE gathers of
// long segments.  Activations are fp16 rows (prepared ones with their
// exponents, or null).
#pragma once
#include "kq_common.h"

// Live problems (M, N > 0); exps[i] per problem.  With `part` room
// (kq_gemm_part_bytes) and the counters, launches that would leave CUs idle run
// in K slices.
bool kq_gemm_eligible(const kq_matmul_problem *ps, int n);
size_t kq_gemm_part_bytes(const kq_matmul_problem *ps, int n);
int kq_gemm_launch(const kq_matmul_problem *ps, const int32_t *const *exps, int n, int y_dtype, uint32_t *counters,
                   float *part, hipStream_t s);

// h = act(x . Wg^T) * (x . Wu^T): `gate` with the up matrix of the same shape
// and row stride.
bool kq_gemm_glu_eligible(const kq_matmul_problem &gate);
int kq_gemm_glu_launch(const kq_matmul_problem &gate, const void *w_up, const int32_t *x_exp, int act, int y_dtype,
                       hipStream_t s);

// The MoE gathers (kq_moe_gather_rows): w1 null for the plain form.  x: x_rows
// fp16 rows; streams: the streaming gather would take the call otherwise.
struct KqGemmGather {
    const char *x;
    const int32_t *x_exp;
    const uint8_t *w0, *w1;
    void *y;
    const int32_t *seg_info, *pair_order;
    const float *b0, *b1;
    int64_t w_expert_bytes, w_row_bytes, y_stride, b_stride;
    uint32_t x_row_bytes, x_bytes;
    int32_t x_pair_div, x_skip, y_skip, N, K, codec, n_pairs, n_experts, y_dtype, act;
    float limit, alpha;
};
bool kq_gemm_gather_eligible(const KqGemmGather &a, int64_t x_rows, int64_t x_row_stride, bool streams);
int kq_gemm_gather_launch(const KqGemmGather &a, hipStream_t s);
