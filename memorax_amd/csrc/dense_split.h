// Internal entry points of dense_split.hip for dense_grads.hip.
#pragma once
#include "common.h"

namespace mrx {

// What a call needs of workspace for the weights as the products read them; 0: not served.  across: for the gradient of the input.
int64_t split_pack_floats(const int64_t *n_out, int layers, int64_t K, bool across);

// y_l = x W_l^T + b_l (outs), or with `dys` instead of x: dx = sum_l dy_l W_l, float32 or bfloat16.
struct SplitCall {
    const float *x = nullptr;
    const void *const *dys = nullptr;
    const void *const *weights = nullptr, *const *biases = nullptr;
    void *const *outs = nullptr;
    const float *residual = nullptr;
    const float *skip = nullptr, *skip_x = nullptr;   // skip[c] skip_x[r][c] is added to the one result
    void *dx = nullptr;
    bool dx_bf16 = false;
    const int64_t *n_out = nullptr;
    int layers = 0;
    int64_t rows = 0, K = 0;
    float *workspace = nullptr;
};
int split_rows(hipStream_t st, const SplitCall &c);

}  // namespace mrx
