// mq_rows.h -- the few-row layers of a Q8_0 BERT encoder (mq_rows.hip).
#pragma once
#include "mq_internal.h"

namespace mq {

constexpr int ROWS_MAX_K = 4096;   // 16 blocks a wave
constexpr int ROWS_MAX_LN = 1024;  // rows formed in registers, their quants in LDS
constexpr int ROWS_MAX_T = 32;     // keys of one query, a lane each; two blocks of the online softmax

enum { ROWS_F32 = 0, ROWS_LN = 1, ROWS_Q = 2 };

struct RowsArgs {
    const void *x_ws = nullptr;  // M rows quantized in the GEMM activation layout, or NULL:
    const float *x = nullptr;    // M dense rows of K floats (16-byte aligned)
    // LayerNorm prologue (res not NULL): the rows are layer_norm(x + res) lw + lb, also stored to
    // xout, which is neither x nor res
    const float *res = nullptr, *lw = nullptr, *lb = nullptr;
    float eps = 0.f;
    float *xout = nullptr;
    const float *bias = nullptr;  // N floats, or NULL
    float *y = nullptr;           // M rows of N floats, ldy apart (no q_out)
    int64_t ldy = 0;
    int M = 0, variant = 0;
    // filled by launch_rows
    const int8_t *wq = nullptr, *xq = nullptr;
    const float *wd = nullptr, *xd = nullptr;
    int8_t *qo = nullptr;
    float *qd = nullptr;
    int64_t m_pad = 0, q_m_pad = 0;
    int n_pad = 0, kch = 0, q_kch = 0, N = 0, K = 0;
};

// y = rows w^T + bias for a prepared Q8_0 weight image of n x k, with the GEMV's sums bit for bit;
// with q_out (LayerNorm prologue only) instead gelu_erf of that, as the Q8_0 activation of the next
// product (the GEMM workspace layout of M rows of n)
hipError_t launch_rows(const void *image, int64_t n, int64_t k, RowsArgs a, void *q_out, hipStream_t s);
// the same of quantized rows (a.x_ws) with the sums of the GEMM at 9 - 32 rows
hipError_t launch_rows_groups(const void *image, int64_t n, int64_t k, RowsArgs a, hipStream_t s);
// full attention over q|k|v rows of 3 H floats (bias added), T at most ROWS_MAX_T, head_dim 32, 64 or
// 128; the rows leave as the Q8_0 activation of the o product in q_out
hipError_t launch_rows_attn(const float *qkv, void *q_out, int variant, int B, int T, int H, int nh, hipStream_t s);
// the most rows that the few-row form takes of a Q8_0 encoder's batches (0: none), and whether it takes
// a batch
int64_t rows_path_limit(int64_t H, int64_t F, int hd);
bool rows_path_fits(int64_t rows, int64_t T, int64_t H, int64_t F, int hd);

}  // namespace mq
