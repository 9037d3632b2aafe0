// Plain local (banded) softmax attention for float32 inputs on the bf16 matrix pipe: forward and gradients
// (src/models/attention/local_attention.py:68-92; the reference takes the gradients from autograd).
//
// v_mfma_f32_16x16x32_bf16 retires 16 times the multiply-adds of the fp32 instruction per cycle.  A float is the sum of
// three bf16 pieces exactly (h + m + l, 24 bits), and a product of two floats is taken as the six piece products above
// 2^-24 of it (h h, h m, m h, m m, h l, l h), accumulated in fp32: as accurate as the fp32 instruction (2-norm against
// float64 at 1300 tokens, windows of 98 and 500: output 1.8e-7 and 3.7e-7, gradients 4.2e-7 and 5.6e-7; 2.4e-7, 4.8e-7,
// 4.6e-7 and 6.6e-7 on the fp32 instruction), at 6 / 16 of its matrix time, and with vector instructions free to run
// beside it, which fp32 MFMAs do not allow.  That holds down to 2^-102: smaller values have pieces below the normal range of
// bf16, which the matrix pipe takes as zero (an output gradient of 1e-30: 4.8e-7; of 1e-36: 4e-4).
// Measured (us, forward / training step; before: the fp32-pipe forward and, for the gradients, the Scatterbrain band kernels
// with zero features on contiguous copies): B=64 L=3136 window 98: 106 / 585 -> 76 / 289; 16 heads of 16384 tokens, window
// 1024: 629 / 3485 -> 432 / 1726; head dim 32, 8 heads of 8192, window 512: 54 / 332 -> 41 / 185.
// The pieces are formed where a tile is staged into LDS (float rows in memory, piece rows in LDS): a preparation pass would
// write and read 1.5 times the inputs again, and the passes are within a small factor of the memory they touch.
//
// A wave owns 16 outer rows (queries; keys when KEYMAJOR) with their operands in registers as pieces and walks 32-row
// tiles of the other side -- short tiles, so that a wave skips what lies outside its own rows' bands.  Products are
// formed transposed (rows = inner, columns = outer): a lane's eight weights of a tile are the contraction slots
// {4 g + i, 16 + 4 g + i} of the second product, whose other operand comes by transposing LDS reads of the same rows.
// Rows are 2 E bytes per piece with 16-byte chunks XOR-swizzled (x3_swz).
//
// Pieces of an infinity are no pieces (inf - inf), a float above the largest bfloat16 becomes one, and piece products of
// values whose product leaves the float range may do so with either sign.  All of that ends in results that are not finite, so a
// wave with such a result takes its rows again with float multiply-adds over the pairs of the band (local_*_plain):
// infinities and NaN then reach what they reach in a float computation over those pairs, at a hundredth of the rate.  The check
// costs 2 % of a training step at window 98 (275 -> 281 us), 1 % at 1024 (1663 -> 1682).
#include "common.h"
#include "local.h"

namespace flyhip {

constexpr int LX_TK = 32, LX_NT = 256;
constexpr float LX_LOG2E = 1.4426950408889634f;

// 32 float rows of E, global -> registers -> three pieces in LDS
template <int E>
struct PieceTile {
    static constexpr int CH = E / 8, TOT = LX_TK * CH, ROWB = 2 * E, PIECE = LX_TK * ROWB, BYTES = 3 * PIECE;
    static_assert(TOT <= LX_NT, "one chunk of eight elements per thread");
    floatx4 r0, r1;
    __device__ __forceinline__ void fetch(const float* src, long stride, int row0, int last_row, int tid) {
        if (TOT == LX_NT || tid < TOT) {
            const float* p = src + (long)min(row0 + tid / CH, last_row) * stride + 8 * (tid % CH);
            r0 = *reinterpret_cast<const floatx4*>(p);
            r1 = *reinterpret_cast<const floatx4*>(p + 4);
        }
    }
    __device__ __forceinline__ void stash(char* dst, int tid) const {
        if (TOT == LX_NT || tid < TOT) {
            const int row = tid / CH;
            uintx4 h, m, l;
            split3(r0, r1, h, m, l);
            char* d = dst + row * ROWB + x3_swz(row, tid % CH, ROWB) * 16;
            *reinterpret_cast<uintx4*>(d) = h;
            *reinterpret_cast<uintx4*>(d + PIECE) = m;
            *reinterpret_cast<uintx4*>(d + 2 * PIECE) = l;
        }
    }
};

// row fragment: elements 32 ks + 8 g .. + 7 of `row`; transposed fragment: column 16 cb + r16 of rows {4 g + i, 16 + 4 g + i}
template <int E>
__device__ __forceinline__ Pieces lx_rows(const char* st, int row, int ks, int g) {
    using PT = PieceTile<E>;
    const char* p = st + row * PT::ROWB + x3_swz(row, 4 * ks + g, PT::ROWB) * 16;
    return Pieces{*reinterpret_cast<const uintx4*>(p), *reinterpret_cast<const uintx4*>(p + PT::PIECE),
                  *reinterpret_cast<const uintx4*>(p + 2 * PT::PIECE)};
}
template <int E>
__device__ __forceinline__ Pieces lx_cols(const char* st, int cb, int r16, int g) {
    using PT = PieceTile<E>;
    const int row = 4 * g + (r16 >> 2), q = r16 & 3;
    const char* p = st + row * PT::ROWB + x3_swz(row, 2 * cb + (q >> 1), PT::ROWB) * 16 + 8 * (q & 1);
    return Pieces{lds_read_tr8(p, p + 16 * PT::ROWB), lds_read_tr8(p + PT::PIECE, p + PT::PIECE + 16 * PT::ROWB),
                  lds_read_tr8(p + 2 * PT::PIECE, p + 2 * PT::PIECE + 16 * PT::ROWB)};
}
__device__ __forceinline__ Pieces lx_load(const float* p) {
    return split<3>(*reinterpret_cast<const floatx4*>(p), *reinterpret_cast<const floatx4*>(p + 4));
}
template <int N>
__device__ __forceinline__ float sum_of(const floatx4 (&x)[N]) {       // (finite only if all of them are)
    floatx4 s = x[0];
#pragma unroll
    for (int j = 1; j < N; ++j) s += x[j];
    return (s[0] + s[1]) + (s[2] + s[3]);
}
__device__ __forceinline__ bool finite_in_wave(float x) { return __builtin_amdgcn_ballot_w64(!(fabsf(x) < INFINITY)) == 0; }
// four lanes per row (lane / 4), E / 4 elements each, in groups of four
template <int E>
struct RowPart {
    floatx4 x[E / 16];
    __device__ __forceinline__ void load(const float* row, int part, float scale = 1.f) {
#pragma unroll
        for (int j = 0; j < E / 16; ++j) x[j] = *reinterpret_cast<const floatx4*>(row + (E / 4) * part + 4 * j) * scale;
    }
    __device__ __forceinline__ float dot(const RowPart& o) const {
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < E / 16; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) d = fmaf(x[j][i], o.x[j][i], d);
        d += __shfl_xor(d, 1);
        return d + __shfl_xor(d, 2);
    }
    __device__ __forceinline__ void add(float w, const RowPart& o) {
#pragma unroll
        for (int j = 0; j < E / 16; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) x[j][i] = fmaf(w, o.x[j][i], x[j][i]);
    }
    __device__ __forceinline__ void store(float* row, int part, float scale) const {
#pragma unroll
        for (int j = 0; j < E / 16; ++j) store4_f32(row + (E / 4) * part + 4 * j, x[j] * scale);
    }
};

// the wave's 16 queries from q0 on, one pass for the largest score and one for the sums
template <int E>
__device__ __forceinline__ void local_fwd_plain(const LocalArgs& a, int b, int h, int q0, int len, int lane) {
    const int part = lane & 3, bh = b * a.H + h, iq = min(q0 + (lane >> 2), a.T - 1);      // (rows past the end do the last one again)
    const float* kptr = reinterpret_cast<const float*>(a.k) + b * a.k_sb + h * a.k_sh;
    const float* vptr = reinterpret_cast<const float*>(a.v) + b * a.v_sb + h * a.v_sh;
    const int lo = max(iq - a.lc / 2, 0), hi = min(iq + (a.lc + 1) / 2, len);
    const float sc = a.temp * LX_LOG2E;
    const uint32_t drop_row = a.drop_thresh != 0u ? drop_row_hash(a.drop_seed, (uint32_t)(bh * a.T + iq)) : 0u;
    RowPart<E> q, y, acc;
    q.load(reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh + (long)iq * a.q_ss, part, sc);            // (scaled before the products: they stay in range longer)
#pragma unroll
    for (int j = 0; j < E / 16; ++j) acc.x[j] = Frag<float>::zero();
    auto score = [&](int n) __attribute__((always_inline)) {
        y.load(kptr + (long)n * a.k_ss, part);
        const float s = q.dot(y), am = a.add_mask ? a.add_mask[(long)iq * a.S + n] : 0.f;
        return am < -1e20f ? -0x1p80f * sc : s + am * sc;
    };
    float m = -1e30f, z = 0.f;
#pragma unroll 1
    for (int n = lo; n < hi; ++n) m = fmaxf(m, score(n));
#pragma unroll 1
    for (int n = lo; n < hi; ++n) {
        const float p = __builtin_amdgcn_exp2f(score(n) - m);
        z += p;
        y.load(vptr + (long)n * a.v_ss, part);
        acc.add(a.drop_thresh == 0u || drop_keep(drop_row, (uint32_t)n, a.drop_thresh) ? p : 0.f, y);
    }
    const bool all_masked = a.add_mask != nullptr && hi > lo && m < -1e20f;
    if (all_masked) z += (float)(a.lc - (hi - lo));
    if (q0 + (lane >> 2) >= a.T) return;
    acc.store(reinterpret_cast<float*>(a.out) + b * a.o_sb + h * a.o_sh + (long)iq * a.o_ss, part,
              (z > 0.f ? 1.0f / z : z == z ? 0.f : z) * (a.drop_thresh != 0u ? a.drop_scale : 1.0f));
    if (a.lse && part == 0) a.lse[(long)bh * a.T + iq] = all_masked ? -INFINITY : z > 0.f ? m * 0.6931471805599453f + __logf(z) : z == z ? 0.f : z;
}

// the gradients of the wave's 16 outer rows from o0 on
template <int E, bool KEYMAJOR>
__device__ __forceinline__ void local_bwd_plain(const LocalBwdArgs& a, int b, int h, int o0, int len, int lane) {
    const int part = lane & 3, bh = b * a.H + h, rows = KEYMAJOR ? a.S : a.T, o = min(o0 + (lane >> 2), rows - 1);
    const float* qptr = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
    const float* kptr = reinterpret_cast<const float*>(a.k) + b * a.k_sb + h * a.k_sh;
    const float* vptr = reinterpret_cast<const float*>(a.v) + b * a.v_sb + h * a.v_sh;
    const float* gptr = reinterpret_cast<const float*>(a.go) + b * a.g_sb + h * a.g_sh;
    const float* y1p = KEYMAJOR ? qptr : kptr;  const long y1s = KEYMAJOR ? a.q_ss : a.k_ss;
    const float* y2p = KEYMAJOR ? gptr : vptr;  const long y2s = KEYMAJOR ? a.g_ss : a.v_ss;
    const int lc_lo = a.lc / 2, lc_hi = (a.lc + 1) / 2;
    const int lo = max(o - (KEYMAJOR ? lc_hi - 1 : lc_lo), 0);
    const int hi = KEYMAJOR ? (o < len ? min(o + lc_lo + 1, a.T) : 0) : min(o + lc_hi, len);
    const float sc = a.temp * LX_LOG2E;
    RowPart<E> x1, x2, y1, y2, acc1, acc2;
    x1.load(KEYMAJOR ? kptr + (long)o * a.k_ss : qptr + (long)o * a.q_ss, part, sc);
    x2.load(KEYMAJOR ? vptr + (long)o * a.v_ss : gptr + (long)o * a.g_ss, part);
    float l_own = 0.f, d_own = 0.f;
    if (!KEYMAJOR) {
        y1.load(reinterpret_cast<const float*>(a.out) + b * a.o_sb + h * a.o_sh + (long)o * a.o_ss, part);
        d_own = x2.dot(y1);
        l_own = a.lse[(long)bh * a.T + o] * LX_LOG2E;
    }
#pragma unroll
    for (int j = 0; j < E / 16; ++j) { acc1.x[j] = Frag<float>::zero(); acc2.x[j] = Frag<float>::zero(); }
#pragma unroll 1
    for (int n = lo; n < hi; ++n) {
        const int i = KEYMAJOR ? n : o, key = KEYMAJOR ? o : n;                     // the pair's query and key
        y1.load(y1p + (long)n * y1s, part);
        y2.load(y2p + (long)n * y2s, part);
        const float s = x1.dot(y1), gv = x2.dot(y2);
        const float lrow = KEYMAJOR ? a.lse[(long)bh * a.T + n] * LX_LOG2E : l_own, drow = KEYMAJOR ? a.delta[(long)bh * a.T + n] : d_own;
        const float am = a.add_mask ? a.add_mask[(long)i * a.S + key] : 0.f;
        const float pr = a.add_mask && lrow == -INFINITY ? 1.0f / (float)a.lc
                                                         : __builtin_amdgcn_exp2f((am < -1e20f ? -0x1p80f * sc : s + am * sc) - lrow);
        float keep = 1.f;
        if (a.drop_thresh != 0u)
            keep = drop_keep(drop_row_hash(a.drop_seed, (uint32_t)(bh * a.T + i)), (uint32_t)key, a.drop_thresh) ? a.drop_scale : 0.f;
        acc1.add(pr * (keep * gv - drow), y1);
        if (KEYMAJOR) acc2.add(pr * keep, y2);
    }
    if (o0 + (lane >> 2) >= rows) return;
    acc1.store(KEYMAJOR ? reinterpret_cast<float*>(a.dk) + b * a.dk_sb + h * a.dk_sh + (long)o * a.dk_ss
                        : reinterpret_cast<float*>(a.dq) + b * a.dq_sb + h * a.dq_sh + (long)o * a.dq_ss, part, a.temp);
    if (KEYMAJOR) acc2.store(reinterpret_cast<float*>(a.dv) + b * a.dv_sb + h * a.dv_sh + (long)o * a.dv_ss, part, 1.f);
}

template <int E>
__global__ __launch_bounds__(LX_NT) void local_fwd_x3_kernel(LocalArgs a) {
    using PT = PieceTile<E>;
    constexpr int KS = E / 32, DB = E / 16, STAGE = 2 * PT::BYTES, TQB = 64;
    extern __shared__ __attribute__((aligned(128))) char lx_smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int n_qt = (a.T + TQB - 1) / TQB;
    const int n_items = a.B * a.H * n_qt;
    const int per_xcd = (n_items + a.n_xcd - 1) / a.n_xcd;
    const int item = (blockIdx.x % a.n_xcd) * per_xcd + blockIdx.x / a.n_xcd;      // neighbouring tiles share a die's L2
    if (item >= n_items) return;                                                    // workgroup-uniform
    const int qt = item % n_qt, bh = item / n_qt, b = bh / a.H, h = bh % a.H;
    const int q0 = qt * TQB, qw0 = q0 + 16 * w;
    const float* qptr = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
    const float* kptr = reinterpret_cast<const float*>(a.k) + b * a.k_sb + h * a.k_sh;
    const float* vptr = reinterpret_cast<const float*>(a.v) + b * a.v_sb + h * a.v_sh;
    const int len = a.lens ? min((int)a.lens[b], a.S) : a.S;
    const int lc_lo = a.lc / 2, lc_hi = (a.lc + 1) / 2;                             // band: -lc_lo <= s - i < lc_hi
    const int q_last = min(q0 + TQB - 1, a.T - 1);
    const int lo = max(0, q0 - lc_lo), hi = min(len, q_last + lc_hi);
    const int kt_lo = lo / LX_TK, kt_hi = (hi > lo) ? (hi + LX_TK - 1) / LX_TK : kt_lo;
    PT rk, rv;
    if (kt_lo < kt_hi) {
        rk.fetch(kptr, a.k_ss, kt_lo * LX_TK, a.S - 1, tid);
        rv.fetch(vptr, a.v_ss, kt_lo * LX_TK, a.S - 1, tid);
    }
    const int iq = qw0 + r16;
    const float* qrow = qptr + (long)min(iq, a.T - 1) * a.q_ss;
    Pieces qp[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qp[ks] = lx_load(qrow + 32 * ks + 8 * g);
    float m_run = -1e30f, ze = 0.f;         // (finite, so that the first rescale is exp2(-huge) = 0 and not inf - inf)
    floatx4 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = Frag<float>::zero();
    const int smin = max(iq - lc_lo, 0);
    const unsigned span = iq < a.T ? (unsigned)max(min(iq + lc_hi, len) - smin, 0) : 0u;
    const uint32_t drop_row = a.drop_thresh != 0u ? drop_row_hash(a.drop_seed, (uint32_t)(bh * a.T + iq)) : 0u;
    const float sc = a.temp * LX_LOG2E;
    if (kt_lo < kt_hi) {
        rk.stash(lx_smem, tid);
        rv.stash(lx_smem + PT::BYTES, tid);
    }
    __syncthreads();
    for (int kt = kt_lo; kt < kt_hi; ++kt) {
        const int s_base = kt * LX_TK, cur = (kt - kt_lo) & 1;
        const char* Ks = lx_smem + cur * STAGE;
        const char* Vs = Ks + PT::BYTES;
        const bool more = kt + 1 < kt_hi;
        if (more) {
            rk.fetch(kptr, a.k_ss, s_base + LX_TK, a.S - 1, tid);
            rv.fetch(vptr, a.v_ss, s_base + LX_TK, a.S - 1, tid);
        }
        // (wave-uniform, scalar) does the tile touch the band of one of the wave's queries; does it lie inside all
        const bool any = !(s_base + LX_TK - 1 - qw0 < -lc_lo || s_base - (qw0 + 15) >= lc_hi || s_base >= len);
        const bool inside = s_base - (qw0 + 15) >= -lc_lo && s_base + LX_TK - 1 - qw0 < lc_hi && s_base + LX_TK <= len &&
                            qw0 + 15 < a.T;
        if (any) {
            floatx4 s[2] = {Frag<float>::zero(), Frag<float>::zero()};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const Pieces kf = lx_rows<E>(Ks, 16 * kb + r16, ks, g);
                    s[kb] = mma_pieces(kf, qp[ks], s[kb]);
                }
            if (a.add_mask) {                                // (uniform)
                const float* am = a.add_mask + (long)min(iq, a.T - 1) * a.S;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int n = s_base + 16 * kb + 4 * g + i;
                        // (an absorbing entry becomes -2^80: its product with the scale is exact, so the multiply-add
                        //  of the exponent below gives exactly 0 for a row whose keys are all hidden)
                        if ((unsigned)(n - smin) < span) s[kb][i] = am[n] < -1e20f ? -0x1p80f : s[kb][i] + am[n];
                    }
            }
            if (!inside) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!((unsigned)(s_base + 16 * kb + 4 * g + i - smin) < span)) s[kb][i] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kb][i]);
            mx = group_max(mx) * sc;
            if (__builtin_amdgcn_ballot_w64(mx > m_run + 8.f) != 0) {
                const float m_new = fmaxf(m_run, mx);
                const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
                m_run = m_new;
                ze *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[kb][i] = __builtin_amdgcn_exp2f(fmaf(s[kb][i], sc, -m_run));      // (masked: -inf, weight 0)
                    ze += s[kb][i];
                }
            if (a.drop_thresh != 0u) {                       // (uniform) dropped weights leave the product, not the denominator
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!drop_keep(drop_row, (uint32_t)(s_base + 16 * kb + 4 * g + i), a.drop_thresh)) s[kb][i] = 0.f;
            }
            const Pieces p = split<3>(s[0], s[1]);
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const Pieces vf = lx_cols<E>(Vs, db, r16, g);
                oacc[db] = mma_pieces(vf, p, oacc[db]);
            }
        }
        if (more) {
            char* nxt = lx_smem + (cur ^ 1) * STAGE;
            rk.stash(nxt, tid);
            rv.stash(nxt + PT::BYTES, tid);
        }
        __syncthreads();
    }
    float z = group_sum(ze);
    // every visible key masked: the positions of the band outside the keys carry the same score in the reference's
    // softmax over the packed band (local_attention.py:68-81), so they count in the denominator
    const bool all_masked = a.add_mask != nullptr && span > 0u && m_run < -1e20f;
    if (all_masked) z += (float)(a.lc - (int)span);
    if (iq < a.T) {
        const float inv = (z > 0.f ? 1.0f / z : 0.f) * (a.drop_thresh != 0u ? a.drop_scale : 1.0f);
        float* optr = reinterpret_cast<float*>(a.out) + b * a.o_sb + h * a.o_sh + (long)iq * a.o_ss;
#pragma unroll
        for (int db = 0; db < DB; ++db) store4_f32(optr + 16 * db + 4 * g, oacc[db] * inv);
        if (a.lse && g == 0)        // a query without visible keys has no pair that would read its entry
            a.lse[((long)b * a.H + h) * a.T + iq] = all_masked ? -INFINITY
                                                        : z > 0.f ? m_run * 0.6931471805599453f + __logf(z) : 0.f;
    }
    if (!finite_in_wave(sum_of(oacc) + ze)) {
        drain_loads();                                      // (the results stored above have gone out)
        local_fwd_plain<E>(a, b, h, qw0, len, lane);
    }
}

// Gradients, in the two orientations of local_bwd_b16_kernel (sblocal.hip): with P_is = exp(t (q_i.k_s + mask) - lse_i) and
// M the kept / (1 - p) mask of a forward with dropout (1 without),
//   query-major: delta_i = g_i.out_i (kept for the other launch), d q_i = t sum_s dS_is k_s,  dS = P (M g.v - delta)
//   key-major:   d k_s = t sum_i dS_is q_i,  d v_s = sum_i M P g_i
template <int E> constexpr size_t local_bwd_x3_smem() { return (size_t)2 * (2 * PieceTile<E>::BYTES + 2 * LX_TK * sizeof(float)); }

// (three workgroups per compute unit, as many as their stages allow, four at 32 dims: the key-major form takes 176 registers of its
// own accord)
template <int E, bool KEYMAJOR>
__global__ __launch_bounds__(LX_NT) __attribute__((amdgpu_waves_per_eu(E == 32 ? 4 : 3, 4))) void local_bwd_x3_kernel(LocalBwdArgs a) {
    using PT = PieceTile<E>;
    constexpr int KS = E / 32, EB = E / 16, STAGE = 2 * PT::BYTES + 2 * LX_TK * (int)sizeof(float), TQB = 64;
    extern __shared__ __attribute__((aligned(128))) char lx_smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int R_out = KEYMAJOR ? a.S : a.T, R_in = KEYMAJOR ? a.T : a.S;
    const int n_ot = (R_out + TQB - 1) / TQB;
    const int n_items = a.B * a.H * n_ot;
    const int per_xcd = (n_items + a.n_xcd - 1) / a.n_xcd;
    const int item = (blockIdx.x % a.n_xcd) * per_xcd + blockIdx.x / a.n_xcd;
    if (item >= n_items) return;                                                    // workgroup-uniform
    const int ot = item % n_ot, bh = item / n_ot, b = bh / a.H, h = bh % a.H;
    const int o0 = ot * TQB, ow0 = o0 + 16 * w, io = ow0 + r16;
    const float* qptr = reinterpret_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
    const float* kptr = reinterpret_cast<const float*>(a.k) + b * a.k_sb + h * a.k_sh;
    const float* vptr = reinterpret_cast<const float*>(a.v) + b * a.v_sb + h * a.v_sh;
    const float* gptr = reinterpret_cast<const float*>(a.go) + b * a.g_sb + h * a.g_sh;
    const float* x1p = KEYMAJOR ? kptr : qptr;  const long x1s = KEYMAJOR ? a.k_ss : a.q_ss;       // outer operands
    const float* x2p = KEYMAJOR ? vptr : gptr;  const long x2s = KEYMAJOR ? a.v_ss : a.g_ss;
    const float* y1p = KEYMAJOR ? qptr : kptr;  const long y1s = KEYMAJOR ? a.q_ss : a.k_ss;       // inner tiles
    const float* y2p = KEYMAJOR ? gptr : vptr;  const long y2s = KEYMAJOR ? a.g_ss : a.v_ss;
    const float* lsep = a.lse + (long)bh * a.T;
    const float* delp = a.delta + (long)bh * a.T;
    const int len = a.lens ? min((int)a.lens[b], a.S) : a.S;
    // the pair (outer o, inner n) is in the band when n - o lies in [-A, Bq), o < Lo and n < Ln
    const int lc_lo = a.lc / 2, lc_hi = (a.lc + 1) / 2;
    const int A = KEYMAJOR ? lc_hi - 1 : lc_lo, Bq = KEYMAJOR ? lc_lo + 1 : lc_hi;
    const int Lo = KEYMAJOR ? len : a.T, Ln = KEYMAJOR ? a.T : len;
    const int o_last = min(min(o0 + TQB - 1, R_out - 1), Lo - 1);
    const int lo = max(0, o0 - A), hi = o_last >= o0 ? min(Ln, o_last + Bq) : 0;
    const int it_lo = lo / LX_TK, it_hi = (hi > lo) ? (hi + LX_TK - 1) / LX_TK : it_lo;
    PT r1, r2;
    float rs = 0.f;                                    // key-major: lse log2e (threads 0 .. 31) and delta (32 .. 63) of the tile's queries
    auto fetch = [&](int it) __attribute__((always_inline)) {
        r1.fetch(y1p, y1s, it * LX_TK, R_in - 1, tid);
        r2.fetch(y2p, y2s, it * LX_TK, R_in - 1, tid);
        if (KEYMAJOR && tid < 2 * LX_TK) {
            const int i = min(it * LX_TK + (tid & (LX_TK - 1)), a.T - 1);
            rs = tid < LX_TK ? lsep[i] * LX_LOG2E : delp[i];
        }
    };
    auto stash = [&](int stage) __attribute__((always_inline)) {
        char* st = lx_smem + stage * STAGE;
        r1.stash(st, tid);
        r2.stash(st + PT::BYTES, tid);
        if (KEYMAJOR && tid < 2 * LX_TK) reinterpret_cast<float*>(st + 2 * PT::BYTES)[tid] = rs;
    };
    if (it_lo < it_hi) fetch(it_lo);

    const long row = min(io, R_out - 1);
    Pieces x1[KS], x2[KS];
    float l_own = 0.f, d_own = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x1[ks] = lx_load(x1p + row * x1s + 32 * ks + 8 * g);
    if (!KEYMAJOR) {
        const float* orow = reinterpret_cast<const float*>(a.out) + b * a.o_sb + h * a.o_sh + row * a.o_ss;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float* gp_ = x2p + row * x2s + 32 * ks + 8 * g;
            const floatx4 g0 = *reinterpret_cast<const floatx4*>(gp_), g1 = *reinterpret_cast<const floatx4*>(gp_ + 4);
            const floatx4 u0 = *reinterpret_cast<const floatx4*>(orow + 32 * ks + 8 * g), u1 = *reinterpret_cast<const floatx4*>(orow + 32 * ks + 8 * g + 4);
            x2[ks] = split<3>(g0, g1);
#pragma unroll
            for (int i = 0; i < 4; ++i) d_own += g0[i] * u0[i] + g1[i] * u1[i];
        }
        d_own = group_sum(d_own);
        if (g == 0 && io < a.T) a.delta[(long)bh * a.T + io] = d_own;
        l_own = lsep[row] * LX_LOG2E;
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) x2[ks] = lx_load(x2p + row * x2s + 32 * ks + 8 * g);
    }
    const int vmin = max(io - A, 0);
    const unsigned vspan = io < Lo ? (unsigned)max(min(io + Bq, Ln) - vmin, 0) : 0u;
    const uint32_t drop_row = (!KEYMAJOR && a.drop_thresh != 0u) ? drop_row_hash(a.drop_seed, (uint32_t)(bh * a.T + io)) : 0u;
    floatx4 acc1[EB], acc2[KEYMAJOR ? EB : 1];
#pragma unroll
    for (int eb = 0; eb < EB; ++eb) acc1[eb] = Frag<float>::zero();
#pragma unroll
    for (int eb = 0; eb < (KEYMAJOR ? EB : 1); ++eb) acc2[eb] = Frag<float>::zero();
    const float sc = a.temp * LX_LOG2E;
    if (it_lo < it_hi) stash(0);
    __syncthreads();
    for (int it = it_lo; it < it_hi; ++it) {
        const int i_base = it * LX_TK, cur = (it - it_lo) & 1;
        const char* Y1 = lx_smem + cur * STAGE;
        const char* Y2 = Y1 + PT::BYTES;
        const float* Ls = reinterpret_cast<const float*>(Y1 + 2 * PT::BYTES);
        const bool more = it + 1 < it_hi;
        if (more) fetch(it + 1);
        // (wave-uniform, scalar) does the tile touch the band of one of the wave's outer rows; does it lie inside all
        const bool any = !(i_base + LX_TK - 1 - ow0 < -A || i_base - (ow0 + 15) >= Bq || i_base >= Ln || ow0 >= Lo);
        const bool inside = i_base - (ow0 + 15) >= -A && i_base + LX_TK - 1 - ow0 < Bq && i_base + LX_TK <= Ln && ow0 + 15 < Lo;
        if (any) {
            floatx4 s[2], gv[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) { s[kb] = Frag<float>::zero(); gv[kb] = Frag<float>::zero(); }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    s[kb] = mma_pieces(lx_rows<E>(Y1, 16 * kb + r16, ks, g), x1[ks], s[kb]);
                    gv[kb] = mma_pieces(lx_rows<E>(Y2, 16 * kb + r16, ks, g), x2[ks], gv[kb]);
                }
            // weights (times M) into s, dS into gv
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                floatx4 ln4, dl4;
                if (KEYMAJOR) {
                    ln4 = *reinterpret_cast<const floatx4*>(Ls + 16 * kb + 4 * g);
                    dl4 = *reinterpret_cast<const floatx4*>(Ls + LX_TK + 16 * kb + 4 * g);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = i_base + 16 * kb + 4 * g + i;
                    const bool ok = inside || (unsigned)(n - vmin) < vspan;
                    const float lrow = KEYMAJOR ? ln4[i] : l_own, drow = KEYMAJOR ? dl4[i] : d_own;
                    float pr = __builtin_amdgcn_exp2f(fmaf(s[kb][i], sc, -lrow));
                    if (a.add_mask) {                        // (uniform) lse = -inf marks a query whose visible keys are all hidden
                        const float am = ok ? a.add_mask[KEYMAJOR ? (long)n * a.S + io : (long)io * a.S + n] : 0.f;
                        pr = lrow == -INFINITY ? 1.0f / (float)a.lc : __builtin_amdgcn_exp2f(fmaf(s[kb][i] + am, sc, -lrow));
                    }
                    if (!ok) pr = 0.f;
                    float keep = 1.f;
                    if (a.drop_thresh != 0u) {               // (uniform)
                        const uint32_t rh = KEYMAJOR ? drop_row_hash(a.drop_seed, (uint32_t)(bh * a.T + n)) : drop_row;
                        keep = drop_keep(rh, (uint32_t)(KEYMAJOR ? io : n), a.drop_thresh) ? a.drop_scale : 0.f;
                    }
                    s[kb][i] = pr * keep;
                    gv[kb][i] = pr * (keep * gv[kb][i] - drow);
                }
            }
            const Pieces ds = split<3>(gv[0], gv[1]);
            Pieces pw;
            if (KEYMAJOR) pw = split<3>(s[0], s[1]);
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) {
                acc1[eb] = mma_pieces(lx_cols<E>(Y1, eb, r16, g), ds, acc1[eb]);
                if (KEYMAJOR) acc2[eb] = mma_pieces(lx_cols<E>(Y2, eb, r16, g), pw, acc2[eb]);
            }
        }
        if (more) stash(cur ^ 1);
        __syncthreads();
    }
    if (io < R_out) {
        float* d1 = KEYMAJOR ? reinterpret_cast<float*>(a.dk) + b * a.dk_sb + h * a.dk_sh + (long)io * a.dk_ss
                             : reinterpret_cast<float*>(a.dq) + b * a.dq_sb + h * a.dq_sh + (long)io * a.dq_ss;
#pragma unroll
        for (int eb = 0; eb < EB; ++eb) store4_f32(d1 + 16 * eb + 4 * g, acc1[eb] * a.temp);
        if (KEYMAJOR) {
            float* d2 = reinterpret_cast<float*>(a.dv) + b * a.dv_sb + h * a.dv_sh + (long)io * a.dv_ss;
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) store4_f32(d2 + 16 * eb + 4 * g, acc2[eb]);
        }
    }
    if (!finite_in_wave(KEYMAJOR ? sum_of(acc1) + sum_of(acc2) : sum_of(acc1))) {
        drain_loads();                                      // (the results stored above have gone out)
        local_bwd_plain<E, KEYMAJOR>(a, b, h, ow0, len, lane);
    }
}

template <int E>
static int launch_fwd(const LocalArgs& a, hipStream_t st) {
    auto kern = local_fwd_x3_kernel<E>;
    constexpr size_t smem = (size_t)4 * PieceTile<E>::BYTES;
    static std::atomic<unsigned long long> lds_set{0};     // (devices on which this kernel has its LDS limit)
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "local_fwd_x3")) return rc;
    const Machine& mach = machine();
    const long items = (long)a.B * a.H * ((a.T + 63) / 64);
    const long grid = (items + mach.xcds - 1) / mach.xcds * mach.xcds;
    if (grid > 2147483647L) return fail(ERR_ARG, "local_fwd: too many workgroups");
    LocalArgs args = a;
    args.n_xcd = mach.xcds;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(LX_NT), smem, st, args);
    return check_launch("local_fwd_x3_kernel");
}
int launch_local_fwd_x3(const LocalArgs& a, int E, hipStream_t st) { return E == 32 ? launch_fwd<32>(a, st) : launch_fwd<64>(a, st); }

template <int E, bool KEYMAJOR>
static int launch_bwd(const LocalBwdArgs& a, hipStream_t st) {
    auto kern = local_bwd_x3_kernel<E, KEYMAJOR>;
    constexpr size_t smem = local_bwd_x3_smem<E>();
    static std::atomic<unsigned long long> lds_set{0};     // (devices on which this kernel has its LDS limit)
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "local_bwd_x3")) return rc;
    const Machine& mach = machine();
    const long items = (long)a.B * a.H * (((KEYMAJOR ? a.S : a.T) + 63) / 64);
    const long grid = (items + mach.xcds - 1) / mach.xcds * mach.xcds;
    if (grid > 2147483647L) return fail(ERR_ARG, "local_bwd: too many workgroups");
    LocalBwdArgs args = a;
    args.n_xcd = mach.xcds;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(LX_NT), smem, st, args);
    return check_launch("local_bwd_x3_kernel");
}
int launch_local_bwd_x3(const LocalBwdArgs& a, int E, hipStream_t st) {
    // (query-major first: it leaves delta for the key-major launch)
    if (E == 32) {
        if (int rc = launch_bwd<32, false>(a, st)) return rc;
        return launch_bwd<32, true>(a, st);
    }
    if (int rc = launch_bwd<64, false>(a, st)) return rc;
    return launch_bwd<64, true>(a, st);
}

}  // namespace flyhip
