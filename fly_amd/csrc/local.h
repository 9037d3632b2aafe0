// The gradients of plain local attention (sblocal.hip) as the exact part of the Scatterbrain-local backward
// (sblocal_far.hip) calls them.
#pragma once
#include "common.h"

namespace flyhip {

struct LocalBwdArgs {
    const void* q; const void* k; const void* v; const void* go; const void* out;
    const float* lse; float* delta;                 // (B, H, T); delta is written by the query-major launch
    const int64_t* lens;
    void* dq; void* dk; void* dv;
    int B, H, T, S, lc;
    long q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, g_sb, g_sh, g_ss, o_sb, o_sh, o_ss;
    long dq_sb, dq_sh, dq_ss, dk_sb, dk_sh, dk_ss, dv_sb, dv_sh, dv_ss;
    float temp;
    int n_xcd;
    // low-rank part of the gradients (B H, rows, E), added to the band's before the results are rounded, or null
    const float* lr_dq = nullptr; const float* lr_dk = nullptr; const float* lr_dv = nullptr;
};

// The exact part of a Scatterbrain-local backward for bfloat16 inputs (band terms with P_is = exp(t q_i.k_s - lse_i), lse =
// the log-normaliser, delta given), the low-rank part lr_dq / lr_dk / lr_dv added before the results are rounded.
int launch_local_bwd_exact(const LocalBwdArgs& a, int E, hipStream_t st);

}  // namespace flyhip
