// Arguments of the projection's backward kernels (fht.hip and fht_bwd.hip).
#pragma once

#include "lffn_common.h"

struct ProjectBwdArgs {
    const float *x;        // [B, H]
    const float *diag;     // [R, J, D]
    const float *z;        // [B, ncols]  (ncols = T*8)
    const float *g_score;  // [B, T]
    float *g_x;            // [R, B, H]
    float *part_d;         // [nblk, R, J, D]
    float *part_b;         // [nblk, R*D]   (columns >= ncols are written as zero)
    int64_t B;
    int H, R, J, T;
    float decay, residual;
    const float *ln_w;     // [H] or null: the projection's input is LayerNorm(x; ln_w, ln_b, ln_eps), formed on
    const float *ln_b;     // load as in the forward; g_x is then the gradient w.r.t. that LayerNorm output
    float ln_eps;
};

// J = 4; logd 8, 9 or 10
__attribute__((visibility("hidden")))
int lffn_internal_project_hash_bwd_mfma(const ProjectBwdArgs &a, int logd, int num_partials, hipStream_t st);
