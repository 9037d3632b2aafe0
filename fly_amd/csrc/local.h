// Plain local attention (local_attention.py:68-92 of the reference): the arguments its kernels share and the launchers that
// cross source files -- sblocal.hip (2-byte inputs, wide heads), local_x3.hip (float32), sblocal_far.hip (the exact part of
// a Scatterbrain-local backward).
#pragma once
#include "common.h"

namespace flyhip {

struct LocalArgs {
    const void* q; const void* k; const void* v; const int64_t* lens; void* out;
    int B, H, T, S, lc;
    long q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss;
    float temp;
    float* lse;                     // optional (B, H, T): log of the softmax denominator, for the backward pass
    int n_xcd;                      // dies the dispatcher deals workgroup ids to (set at launch)
    // dropout of the probabilities (drop_thresh != 0): pair (query i, key s) of (b, h) is kept when the hash of
    // (seed, row = (b H + h) T + i, s) reaches the threshold, and scaled by 1 / (1 - p); the denominator sums all
    uint32_t drop_seed, drop_thresh; float drop_scale;
    // optional additive mask (T, S), float32, rows contiguous: added to q.k before the temperature.  Entries of -1e24
    // absorb the product (every masked score is the same float), so a query whose visible keys are all masked gets
    // equal weights 1 / local_context -- over the positions of its band that fall outside the keys as well, which
    // count in the denominator only; its lse entry is -inf, the marker the backward kernel reads.
    const float* add_mask;
};

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
    // float32 only: the forward's additive mask and dropout (see LocalArgs)
    const float* add_mask = nullptr;
    uint32_t drop_seed = 0, drop_thresh = 0; float drop_scale = 1.f;
};

// The exact part of a Scatterbrain-local backward for bfloat16 inputs (band terms with P_is = exp(t q_i.k_s - lse_i), lse =
// the log-normaliser, delta given), the low-rank part lr_dq / lr_dk / lr_dv added before the results are rounded.
int launch_local_bwd_exact(const LocalBwdArgs& a, int E, hipStream_t st);

// float32 inputs, head dims 32 and 64, every product from three bf16 pieces per operand
int launch_local_fwd_x3(const LocalArgs& a, int E, hipStream_t st);
int launch_local_bwd_x3(const LocalBwdArgs& a, int E, hipStream_t st);

}  // namespace flyhip
