// The low-rank part of the Scatterbrain-local backward for bfloat16 inputs, without the "all keys minus the band" of
// the kernels in sblocal_prep.hip.
//
// The reference obtains these gradients from autograd through softmax_kernel (src/models/attention/feature_maps_sb.py:51-82)
// and sblocal_attention.py:73-122.  With psi_i = Phi(q_i) exp(kappa) / Z_i, phi_s = Phi(k_s) exp(-kappa), c_i = g_i.out_i and
// df_is = g_i.v_s - c_i, a pair outside the band has the weight psi_i.phi_s, so
//   u_i  = psi_i o sum_{s outside} df_is phi_s        (gradient w.r.t. the log-features of q_i)
//   uk_s = phi_s o sum_{i outside} df_is psi_i,   d v_s += sum_{i outside} (psi_i.phi_s) g_i
// and inside the band the gradient is that of plain local attention with log Z in the place of its log-denominator.
// Rows are taken in chunks of 64.  Seen from a chunk, every chunk of the other side is
//   inside  the band for all pairs    -- no low-rank work at all (the kernels that subtract the band's part spend
//                                        M-wide products on every pair of it: 15 of 17 chunks at a window of 1024),
//   far     no pair in the band       -- through the sums  KV_c = sum phi v^T, sum phi  (QG_c = sum psi g^T, sum psi c) of the
//                                        chunks, kept as prefix sums: the chunks before the window are one of them, those
//                                        after it the sum over all chunks minus the one that ends with the window,
//   an edge some pairs in the band    -- the pairs outside it one by one (two chunks at a window that is a multiple of 128,
//                                        up to four otherwise).
// The difference is taken in float32, so the chunks after the window carry 2^-24 of the sum over all chunks; the pairs of the
// band enter no product and are not subtracted one by one.
// What float32 would hold stays in that precision: far sums, df, low-rank weights, the gradients of the log-features and the
// band's P and dS enter the products as three bf16 pieces (exactly), features as three with more than 128 of them, else as
// two (2^-17, as in the kernels in sblocal_prep.hip).  Against float64 on the same output and log-normaliser, over 28 problems of
// 4 to 32 heads, windows of 12 to 1024: 2-norm error of the bfloat16 gradients 1.5e-3 to 1.9e-3, the rounding of the results,
// and 0.04 to 0.08 % of them rounded otherwise with 256 features (library products in float32: 0.03 to 0.2 %), 0.06 to 0.4 %
// with fewer (the kernels in sblocal_prep.hip: 0.08 to 0.6 %).  Two pieces throughout took 1860 us a step instead of 2130 and
// rounded 0.1 to 0.45 % otherwise with 256 features.
//
//   far_chunk_kernel    KV_c and QG_c summed over the chunks of a segment, every prefix of it kept, stabilised by the largest
//                       log-feature so far
//   far_scan_kernel     inclusive prefix sums over the segments in common units, in place of their last chunks' sums
//   far_lowrank_kernel  query-major and key-major: far and edge terms, chain rule through the feature map -> float32
//   local_bwd_b16_kernel<EXACT> (sblocal.hip)  the band, plus the low-rank part, rounded once
//
// Measured at B=1, H=16, L=16384, window 1024, 256 features, where the backward ran as library products over windows of
// keys before (20.8 ms): chunks 203, scan 19, low-rank 345 (query-major) and 752 (key-major), band 223 and 337 us.  The
// chunk sums (66 KB per 64 rows and side at 256 features) bound the first two: a scan over every chunk instead of every
// segment moved 1.1 GB in 225 us.  The low-rank kernels wait for the far sums (five trips to the cache), and the key-major one
// spends most of its time on the edges: their features, the weights of their pairs and the pieces of both (matrix pipe 26 %,
// vector ALU 36 %, LDS 27 % of its cycles at two waves per SIMD, which wait for memory or a barrier 47 % of theirs).
#include "common.h"
#include "local.h"
#include <algorithm>

namespace flyhip {

constexpr int FC = 64;                              // rows per chunk
struct FarArgs {
    const uint16_t* q; const uint16_t* k; const uint16_t* v; const uint16_t* go; const uint16_t* out;
    const float* ln; const float* proj; const int64_t* lens;
    float* c;                                       // (BH, T): g . out
    float* kscale; float* qscale;                   // (BH, chunks): base-2 log of the units a chunk's sums are kept in
    float* kv; float* qg;                           // (BH, chunks, M (E + 1)): prefix sums [M][E] | [M], see FarPrefix
    float* dq; float* dk; float* dv;                // low-rank part of the gradients, (BH, rows, E)
    int B, H, T, S, lc, mh_valid, n_kc, n_qc;
    int seg;                                        // chunks whose sums one workgroup adds up
    long q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, g_sb, g_sh, g_ss, o_sb, o_sh, o_ss;
    float temp;
    int n_xcd;
};

constexpr float FAR_LOG2E = 1.4426950408889634f;
// bf16 pieces a feature enters the products in (everything else but the bfloat16 tensors themselves: three)
constexpr int far_pieces_of(int M) { return M > 128 ? 3 : 2; }

// largest unit of the keys of a (batch, head) (base 2; 0 when no key is valid).  red: NW floats; ends with a barrier.
template <int NT>
__device__ __forceinline__ float far_kappa(const FarArgs& a, int bh, float* red, int tid) {
    float m = -INFINITY;
    for (int i = tid; i < a.n_kc; i += NT) m = fmaxf(m, a.kscale[(long)bh * a.n_kc + i]);
    m = wave_max(m);
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int i = 1; i < NT / 64; ++i) m = fmaxf(m, red[i]);
    __syncthreads();
    return m == -INFINITY ? 0.f : m;
}

// 64 rows of one side on their way into LDS: x (the rows that have features) and y (values, or output gradients) row-major
// with padded rows; diag = t log2e |x|^2 / 2, ext = the rest of the row's log-feature bias (-inf: no such row), cs = c
template <int E, int NT>
struct FarTile {
    static constexpr int LD = E + 8;
    Tile16<FC, E, NT> x, y;
    float ext, cv;
    // queries: bias base + kappa - log Z; keys: base - kappa.  base = -log2(2 mh) / 2
    __device__ __forceinline__ void fetch(const FarArgs& a, bool queries, const uint16_t* xp, long xs, const uint16_t* yp, long ys,
                                          int bh, int row0, int len, float base, float kappa, int tid) {
        const int last = (queries ? a.T : a.S) - 1;
        x.fetch(xp, xs, row0, last, tid);
        y.fetch(yp, ys, row0, last, tid);
        ext = -INFINITY;
        cv = 0.f;
        if (tid < FC && row0 + tid < len) {
            const long at = (long)bh * a.T + row0 + tid;
            ext = queries ? base + kappa - a.ln[at] * FAR_LOG2E : base - kappa;
            if (queries && a.c) cv = a.c[at];
        }
    }
    __device__ __forceinline__ void stash(const FarArgs& a, uint16_t* Xs, uint16_t* Ys, float* diag, float* exts, float* cs, int tid) const {
        x.template stash<LD>(Xs, tid);
        y.template stash<LD>(Ys, tid);
        constexpr int C8 = E / 8;
#pragma unroll
        for (int j = 0; j < Tile16<FC, E, NT>::N; ++j) {
            const int idx = tid + NT * j;
            float sq = 0.f;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const float lo = __uint_as_float(x.r[j][n] << 16), hi = __uint_as_float(x.r[j][n] & 0xffff0000u);
                sq += lo * lo + hi * hi;
            }
#pragma unroll
            for (int off = 1; off < C8; off <<= 1) sq += __shfl_xor(sq, off);          // the C8 lanes of a row
            if (idx % C8 == 0 && idx < FC * C8) diag[idx / C8] = 0.5f * a.temp * FAR_LOG2E * sq;
        }
        if (tid < FC) { exts[tid] = ext; cs[tid] = cv; }
    }
};

// this wave's 16 rows of sqrt(t) log2e P in three bf16 pieces (exact): lane (r16, g) holds columns 32 ks + 8 g .. + 7 of row r16
template <int KS>
struct FarProj {
    Pieces p[KS];
    __device__ __forceinline__ void load(const float* proj, int row, int E, float scale, int g) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float* src = proj + (long)row * E + 32 * ks + 8 * g;
            p[ks] = split<3>(*reinterpret_cast<const floatx4*>(src) * scale, *reinterpret_cast<const floatx4*>(src + 4) * scale);
        }
    }
    // rows of x . P^T: result rows = rows of x, columns (lane r16) = rows of P
    __device__ __forceinline__ floatx4 rows_by_features(const uint16_t* x0) const {
        floatx4 d = Frag<float>::zero();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) d = mma_pieces(*reinterpret_cast<const uintx4*>(x0 + 32 * ks), p[ks], d);
        return d;
    }
    // the same transposed: result rows = rows of P, columns = rows of x
    __device__ __forceinline__ floatx4 features_by_rows(const uint16_t* x0) const {
        floatx4 d = Frag<float>::zero();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) d = mma_pieces(p[ks], *reinterpret_cast<const uintx4*>(x0 + 32 * ks), d);
        return d;
    }
};

// ---------------------------------------------------------------------------------------
// sums of the chunks
// ---------------------------------------------------------------------------------------
// A segment of `seg` chunks per workgroup, 16 projection rows (32 features, exp(+.) and exp(-.)) per wave.  The projection
// is formed with a chunk's rows as result rows, which leaves a lane with one feature of 16 rows: the operand of F^T Y as it
// stands.  The sums stay in the accumulators from chunk to chunk and are written after each: the prefix sum inside the
// segment, in units of the largest log-feature so far (a whole power of two, so that moving to a larger one is exact).
// The scan then has the segments' last chunks to read and write instead of every one.
template <int E, int M>
__global__ __launch_bounds__(2 * M) void far_chunk_kernel(FarArgs a) {
    constexpr int NW = M / 32, NT = 64 * NW, MH = M / 2, KS = E / 32, EB = E / 16, LD = E + 8, PER = M * (E + 1);
    __shared__ __attribute__((aligned(16))) uint16_t Xs[FC * LD], Ys[FC * LD];
    __shared__ __attribute__((aligned(16))) float diag[FC], exts[FC], cs[FC];
    __shared__ float red[NW];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
    const int k_segs = (a.n_kc + a.seg - 1) / a.seg;
    const bool queries = (int)blockIdx.x >= k_segs;
    const int n_c = queries ? a.n_qc : a.n_kc;
    const int c_lo = (queries ? blockIdx.x - k_segs : blockIdx.x) * a.seg, c_hi = min(c_lo + a.seg, n_c);
    const int len = queries ? a.T : (a.lens ? min((int)a.lens[b], a.S) : a.S);
    const uint16_t* xp = queries ? a.q + b * a.q_sb + h * a.q_sh : a.k + b * a.k_sb + h * a.k_sh;
    const uint16_t* yp = queries ? a.go + b * a.g_sb + h * a.g_sh : a.v + b * a.v_sb + h * a.v_sh;
    const long xs = queries ? a.q_ss : a.k_ss, ys = queries ? a.g_ss : a.v_ss;
    FarTile<E, NT> t;
    Tile16<FC, E, NT> o;
    FarArgs na = a;
    na.c = nullptr;                                 // (formed here)
    const float base = -0.5f * __log2f(2.0f * a.mh_valid);
    const uint16_t* op = a.out + b * a.o_sb + h * a.o_sh;
    t.fetch(na, queries, xp, xs, yp, ys, bh, c_lo * FC, len, base, 0.f, tid);
    if (queries) o.fetch(op, a.o_ss, c_lo * FC, a.T - 1, tid);
    FarProj<KS> P;
    P.load(a.proj, 16 * w + r16, E, sqrtf(a.temp) * FAR_LOG2E, g);
    const bool fvalid = 16 * w + r16 < a.mh_valid;
    floatx4 acc[2][EB];
    float tot[2] = {0.f, 0.f}, unit = -INFINITY;
#pragma unroll
    for (int sg = 0; sg < 2; ++sg)
#pragma unroll
        for (int eb = 0; eb < EB; ++eb) acc[sg][eb] = Frag<float>::zero();
#pragma unroll 1
    for (int c = c_lo; c < c_hi; ++c) {
        t.stash(a, Xs, Ys, diag, exts, cs, tid);
        if (queries) {
            // c = g . out, C8 lanes per row
            constexpr int C8 = E / 8;
            __syncthreads();                        // (cs was zeroed by stash)
#pragma unroll
            for (int j = 0; j < Tile16<FC, E, NT>::N; ++j) {
                const int idx = tid + NT * j, row = idx / C8;
                float d = 0.f;
#pragma unroll
                for (int n = 0; n < 4; ++n)
                    d += __uint_as_float(o.r[j][n] << 16) * __uint_as_float(t.y.r[j][n] << 16) +
                         __uint_as_float(o.r[j][n] & 0xffff0000u) * __uint_as_float(t.y.r[j][n] & 0xffff0000u);
#pragma unroll
                for (int off = 1; off < C8; off <<= 1) d += __shfl_xor(d, off);
                if (idx % C8 == 0 && idx < FC * C8) {
                    cs[row] = d;
                    if (c * FC + row < a.T) a.c[(long)bh * a.T + c * FC + row] = d;
                }
            }
        }
        if (c + 1 < c_hi) {                         // (workgroup-uniform)
            t.fetch(na, queries, xp, xs, yp, ys, bh, (c + 1) * FC, len, base, 0.f, tid);
            if (queries) o.fetch(op, a.o_ss, (c + 1) * FC, a.T - 1, tid);
        }
        __syncthreads();

        floatx4 dd[4];
        float mx = -INFINITY;
        auto bias_of = [&](int kb) __attribute__((always_inline)) {
            return *reinterpret_cast<const floatx4*>(exts + 16 * kb + 4 * g) - *reinterpret_cast<const floatx4*>(diag + 16 * kb + 4 * g);
        };
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            dd[kb] = P.rows_by_features(Xs + (16 * kb + r16) * LD + 8 * g);
            const floatx4 bias = bias_of(kb);
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, fvalid ? fabsf(dd[kb][i]) + bias[i] : -INFINITY);
        }
        mx = wave_max(mx);
        if (lane == 0) red[w] = mx;
        __syncthreads();
        const float before = unit;
#pragma unroll
        for (int i = 0; i < NW; ++i) unit = fmaxf(unit, ceilf(red[i]));
        if (tid == 0) (queries ? a.qscale : a.kscale)[(long)bh * n_c + c] = unit;
        const float shift = unit == -INFINITY ? 0.f : unit;
        if (unit > before && before != -INFINITY) { // (workgroup-uniform; sums in other units before)
            const float f = __builtin_amdgcn_exp2f(before - unit);
#pragma unroll
            for (int sg = 0; sg < 2; ++sg) {
                tot[sg] *= f;
#pragma unroll
                for (int eb = 0; eb < EB; ++eb) acc[sg][eb] *= f;
            }
        }
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
            PiecesOf<far_pieces_of(M)> fp[2];
#pragma unroll
            for (int sg = 0; sg < 2; ++sg) {
                floatx4 f[2];
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    const int kb = 2 * t2 + hb;
                    const floatx4 wr = *reinterpret_cast<const floatx4*>(cs + 16 * kb + 4 * g);
                    const floatx4 bias = bias_of(kb);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float x = __builtin_amdgcn_exp2f((sg ? -dd[kb][i] : dd[kb][i]) + bias[i] - shift);
                        f[hb][i] = fvalid ? x : 0.f;
                        tot[sg] += queries ? f[hb][i] * wr[i] : f[hb][i];
                    }
                }
                fp[sg] = split<far_pieces_of(M)>(f[0], f[1]);
            }
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) {
                const uint16_t* yq = Ys + (32 * t2 + 4 * g + (r16 >> 2)) * LD + 16 * eb + 4 * (r16 & 3);
                const uintx4 yt = lds_read_tr8(reinterpret_cast<const char*>(yq), reinterpret_cast<const char*>(yq + 16 * LD));
#pragma unroll
                for (int sg = 0; sg < 2; ++sg)                          // (transposed: a lane's results are four columns of one feature)
                    acc[sg][eb] = mma_pieces(yt, fp[sg], acc[sg][eb]);
            }
        }
        float* dst = (queries ? a.qg : a.kv) + ((long)bh * n_c + c) * PER;
        const uint32_t lane_at = (uint32_t)((16 * w + r16) * E + 4 * g);
#pragma unroll
        for (int sg = 0; sg < 2; ++sg) {
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) *reinterpret_cast<floatx4*>(dst + sg * MH * E + lane_at + 16 * eb) = acc[sg][eb];
            const float s = group_sum(tot[sg]);
            if (g == 0) dst[M * E + sg * MH + 16 * w + r16] = s;
        }
        __syncthreads();                            // the tiles are free
    }
}

// inclusive prefix sums over the segments of a (batch, head), in place of the sums of their last chunks, in the common
// units of the features (exp(kappa) taken out of the keys and put into the queries); eight loads in flight per thread
constexpr int FAR_SCAN_NT = 256;
__global__ __launch_bounds__(FAR_SCAN_NT) void far_scan_kernel(FarArgs a, int per4) {
    __shared__ float red[FAR_SCAN_NT / 64];
    const int bh = blockIdx.z, e = blockIdx.x * FAR_SCAN_NT + threadIdx.x;
    const bool queries = blockIdx.y != 0;
    const float kappa = far_kappa<FAR_SCAN_NT>(a, bh, red, threadIdx.x);
    if (e >= per4) return;
    const int n_c = queries ? a.n_qc : a.n_kc, n = (n_c + a.seg - 1) / a.seg;
    const float* unit = (queries ? a.qscale : a.kscale) + (long)bh * n_c;
    const float ref = queries ? kappa : -kappa;
    floatx4* p = reinterpret_cast<floatx4*>(queries ? a.qg : a.kv) + (long)bh * n_c * per4 + e;
    floatx4 run = Frag<float>::zero();
    for (int s0 = 0; s0 < n; s0 += 8) {
        floatx4 x[8];
        int at[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            at[j] = min((s0 + j + 1) * a.seg, n_c) - 1;     // (past the end: the last chunk, not used)
            x[j] = p[(long)at[j] * per4];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (s0 + j < n) {
                run += x[j] * __builtin_amdgcn_exp2f(unit[at[j]] + ref);
                p[(long)at[j] * per4] = run;
            }
    }
}

// the sum over the chunks 0 .. c of a (batch, head) in common units, from what the two kernels above leave: at a
// segment's last chunk as it stands, elsewhere the previous segment's end plus the prefix sum inside the segment
struct FarPrefix {
    const float* whole = nullptr; const float* part = nullptr;
    float f = 0.f;
    __device__ __forceinline__ FarPrefix(const float* sums, const float* unit, float ref, long per, int c, int n_c, int seg) {
        if (c < 0) return;                          // (no chunk: 0)
        const int s = c / seg;
        if (c == min((s + 1) * seg, n_c) - 1) { whole = sums + c * per; return; }
        if (s > 0) whole = sums + ((long)s * seg - 1) * per;
        part = sums + c * per;
        f = __builtin_amdgcn_exp2f(unit[c] + ref);
    }
    // x[j] += sign * (the four entries from at(j) on), all loads of a source in flight together (the branches are uniform)
    template <int N, typename At>
    __device__ __forceinline__ void add(floatx4 (&x)[N], float sign, At at) const {
        if (whole) {
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] += *reinterpret_cast<const floatx4*>(whole + at(j)) * sign;
        }
        if (part) {
            const float fs = sign * f;
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] += *reinterpret_cast<const floatx4*>(part + at(j)) * fs;
        }
    }
};

// ---------------------------------------------------------------------------------------
// far and edge terms of 64 outer rows
// ---------------------------------------------------------------------------------------
// 16 projection rows (32 features) per wave, all 64 outer rows: every feature of an edge chunk is formed once per
// workgroup and goes from registers into the products.  Sums over features (chain rule, d v) are per wave until the end.
// Key-major needs two operands transposed as well, the far sums and the edge features: it takes them by transposing LDS reads
// of what it has, not by strided loads and a second evaluation (730 -> 600 us at the size above with operands in two pieces;
// 752 as they are now).  The pieces go through one buffer per wave in turn: side by side they would leave one workgroup per
// compute unit at 128 features, and no room at 256 for the own features' smaller pieces, which do not fit the registers.
// columns of the result reduced over the waves at a time: two 16-column blocks where that takes no more LDS
template <int M, bool KEYMAJOR>
constexpr size_t far_reduce_cols() { return KEYMAJOR || M < 256 ? 32 : 16; }
constexpr int FAR_LDT = 32 + 8;                                                     // row stride of the transposed features, key-major
// bytes of the region that holds, one after the other, the waves' far rows (key-major, one piece at a time), the inner chunk
// with df and (key-major, one piece at a time) the waves' transposed features, the reduction
template <int E, int M, bool KEYMAJOR>
constexpr size_t far_lowrank_shared() {
    size_t n = (size_t)2 * FC * (E + 8) * 2 + 3 * 8 * 64 * 16 + (KEYMAJOR ? (size_t)(M / 32) * 32 * FAR_LDT * 2 : 0);
    const size_t red = far_reduce_cols<M, KEYMAJOR>() * (M / 32) * FC * 4, rows = KEYMAJOR ? (size_t)(M / 32) * 32 * (E + 8) * 2 : 0;
    if (n < red) n = red;
    return n < rows ? rows : n;
}
// key-major: the second and third pieces of the outer rows' features, where the registers do not hold them
template <int M, bool KEYMAJOR>
constexpr size_t far_own_pieces() { return KEYMAJOR && far_pieces_of(M) == 3 ? (size_t)(M / 32) * 2 * 4 * 64 * 16 : 0; }
template <int E, int M, bool KEYMAJOR>
constexpr size_t far_lowrank_smem() {
    return (size_t)2 * FC * (E + 8) * 2 + far_lowrank_shared<E, M, KEYMAJOR>() + far_own_pieces<M, KEYMAJOR>() +
           sizeof(float) * (6 * FC + (M / 32) * (FC + 1) + 3) / 16 * 16;
}

template <int E, int M, bool KEYMAJOR>
__global__ __launch_bounds__(2 * M) __attribute__((amdgpu_waves_per_eu(!KEYMAJOR && M >= 256 ? 4 : 2, !KEYMAJOR && M >= 256 ? 8 : 2))) void far_lowrank_kernel(FarArgs a) {
    constexpr int NW = M / 32, NT = 64 * NW, MH = M / 2, KS = E / 32, EB = E / 16, LD = E + 8, PER = M * (E + 1);
    constexpr size_t TILES = (size_t)2 * FC * LD * 2;
    constexpr int NF = far_pieces_of(M), NR = NF == 3 ? 1 : NF;                      // pieces of a feature; of the own ones, in registers
    extern __shared__ __attribute__((aligned(128))) char far_smem[];
    uint16_t* Xo = reinterpret_cast<uint16_t*>(far_smem);
    uint16_t* Yo = Xo + FC * LD;
    uint16_t* Xi = Yo + FC * LD;                                                    // inner chunk, then df; the reduction overlays both
    uint16_t* Yi = Xi + FC * LD;
    uintx4* DF = reinterpret_cast<uintx4*>(Yi + FC * LD);                           // [piece][step, outer block][lane]
    float* red = reinterpret_cast<float*>(Xi);
    char* after = far_smem + TILES + far_lowrank_shared<E, M, KEYMAJOR>();
    float* diago = reinterpret_cast<float*>(after + far_own_pieces<M, KEYMAJOR>());
    float* exto = diago + FC; float* co = exto + FC;
    float* diagi = co + FC; float* exti = diagi + FC; float* ci = exti + FC;
    float* us = ci + FC;                                                            // [NW][FC]
    float* kred = us + NW * FC;                                                     // [NW]
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    uintx4* FO = reinterpret_cast<uintx4*>(after) + w * 2 * 4 * 64 + lane;          // [piece - 1][outer block][lane], see own_pieces
    // key-major: one piece of the wave's features of 32 inner rows, [sign, 16 features][rows]
    uint16_t* ft = reinterpret_cast<uint16_t*>(DF + 3 * 8 * 64) + w * 32 * FAR_LDT;
    const int Lo = KEYMAJOR ? a.S : a.T;
    const int n_oc = KEYMAJOR ? a.n_kc : a.n_qc, n_ic = KEYMAJOR ? a.n_qc : a.n_kc;
    const int n_items = a.B * a.H * n_oc;
    const int per_xcd = (n_items + a.n_xcd - 1) / a.n_xcd;
    const int item = (blockIdx.x % a.n_xcd) * per_xcd + blockIdx.x / a.n_xcd;      // neighbouring tiles share a die's L2
    if (item >= n_items) return;                                                    // workgroup-uniform
    const int oc = item % n_oc, bh = item / n_oc, b = bh / a.H, h = bh % a.H;
    const int o0 = oc * FC;
    const int klen = a.lens ? min((int)a.lens[b], a.S) : a.S;
    const int len_o = KEYMAJOR ? klen : a.T, len_i = KEYMAJOR ? a.T : klen;
    const uint16_t* qp = a.q + b * a.q_sb + h * a.q_sh;
    const uint16_t* kp = a.k + b * a.k_sb + h * a.k_sh;
    const uint16_t* vp = a.v + b * a.v_sb + h * a.v_sh;
    const uint16_t* gp = a.go + b * a.g_sb + h * a.g_sh;
    const uint16_t* xop = KEYMAJOR ? kp : qp; const uint16_t* yop = KEYMAJOR ? vp : gp;
    const uint16_t* xip = KEYMAJOR ? qp : kp; const uint16_t* yip = KEYMAJOR ? gp : vp;
    const long xos = KEYMAJOR ? a.k_ss : a.q_ss, yos = KEYMAJOR ? a.v_ss : a.g_ss;
    const long xis = KEYMAJOR ? a.q_ss : a.k_ss, yis = KEYMAJOR ? a.g_ss : a.v_ss;
    // the pair (outer o, inner n) is in the band when n - o lies in [-A, Bq)
    const int lc_lo = a.lc / 2, lc_hi = (a.lc + 1) / 2;
    const int A = KEYMAJOR ? lc_hi - 1 : lc_lo, Bq = KEYMAJOR ? lc_lo + 1 : lc_hi;
    // inner chunks [c0, c1) meet the band of some row; [e0, e1) lie inside the band of every row; the rest are far
    const int c0 = min(n_ic, max(0, o0 - A) / FC);
    const int c1 = max(c0, min(n_ic, (max(0, o0 + FC - 1 + Bq) + FC - 1) / FC));
    const int e0 = min(c1, max(c0, (max(0, o0 + FC - 1 - A) + FC - 1) / FC));
    const int e1 = max(e0, min(c1, max(0, o0 + Bq) / FC));

    const float base = -0.5f * __log2f(2.0f * a.mh_valid);
    const float kappa = far_kappa<NT>(a, bh, kred, tid);
    FarTile<E, NT> t;
    t.fetch(a, !KEYMAJOR, xop, xos, yop, yos, bh, o0, len_o, base, kappa, tid);
    FarProj<KS> P;
    P.load(a.proj, 16 * w + r16, E, sqrtf(a.temp) * FAR_LOG2E, g);
    t.stash(a, Xo, Yo, diago, exto, co, tid);
    int ic = c0 < e0 ? c0 : e1;                                                     // edges: c0 .. e0 - 1, e1 .. c1 - 1
    constexpr bool AHEAD = !KEYMAJOR || NW >= 4;                                    // (registers for the next chunk's rows)
    if (AHEAD && ic < c1) t.fetch(a, KEYMAJOR, xip, xis, yip, yis, bh, ic * FC, len_i, base, kappa, tid);
    __syncthreads();

    // own features: result rows = features 16 w + 4 g + i (sign sg), columns = outer rows 16 ob + r16
    auto own_features = [&](int ob, floatx4& f0, floatx4& f1) __attribute__((always_inline)) {
        const floatx4 dd = P.features_by_rows(Xo + (16 * ob + r16) * LD + 8 * g);
        const float bias = exto[16 * ob + r16] - diago[16 * ob + r16];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool ok = 16 * w + 4 * g + i < a.mh_valid;
            f0[i] = ok ? __builtin_amdgcn_exp2f(bias + dd[i]) : 0.f;
            f1[i] = ok ? __builtin_amdgcn_exp2f(bias - dd[i]) : 0.f;
        }
    };
    // key-major: needed throughout, as operands with slots (sg, 4 g + i); query-major: formed where they are used
    PiecesOf<NR> fo[KEYMAJOR ? 4 : 1];
    auto own_pieces = [&](int ob) __attribute__((always_inline)) {
        PiecesOf<NF> r;
#pragma unroll
        for (int pc = 0; pc < NF; ++pc) r.p[pc] = pc < NR ? fo[KEYMAJOR ? ob : 0].p[pc < NR ? pc : 0] : FO[(4 * (pc - 1) + ob) * 64];
        return r;
    };
    if (KEYMAJOR) {
#pragma unroll
        for (int ob = 0; ob < 4; ++ob) {
            floatx4 f0, f1;
            own_features(ob, f0, f1);
            const PiecesOf<NF> f = split<NF>(f0, f1);
#pragma unroll
            for (int pc = 0; pc < NF; ++pc) {
                if (pc < NR) fo[KEYMAJOR ? ob : 0].p[pc < NR ? pc : 0] = f.p[pc];
                else FO[(4 * (pc - 1) + ob) * 64] = f.p[pc];                        // (read back by the same lane only)
            }
        }
    }

    // far terms from the prefix sums of the inner side: pre(c0) + (all - pre(c1))
    const float* pre = (KEYMAJOR ? a.qg : a.kv) + (long)bh * n_ic * PER;
    const float* units = (KEYMAJOR ? a.qscale : a.kscale) + (long)bh * n_ic;
    const float ref = KEYMAJOR ? kappa : -kappa;
    const FarPrefix p0(pre, units, ref, PER, c0 - 1, n_ic, a.seg);
    const FarPrefix p1(pre, units, ref, PER, c1 < n_ic ? c1 - 1 : -1, n_ic, a.seg);
    const FarPrefix pn(pre, units, ref, PER, c1 < n_ic ? n_ic - 1 : -1, n_ic, a.seg);
    // (every load of a source in flight together: a source is one trip to the cache, and nothing else hides it)
    floatx4 fx[2 * (2 * KS + 1)];                                                   // [sign][row: 32 ks + 8 g .. + 7 | features 4 g .. + 3]
#pragma unroll
    for (int j = 0; j < 2 * (2 * KS + 1); ++j) fx[j] = Frag<float>::zero();
    {
        const uint32_t row_at = (uint32_t)((16 * w + r16) * E + 8 * g), vec_at = (uint32_t)(16 * w + 4 * g);
        auto at = [&](int j) __attribute__((always_inline)) {
            const int sg = j / (2 * KS + 1), n = j % (2 * KS + 1);
            return n < 2 * KS ? row_at + sg * MH * E + 32 * (n >> 1) + 4 * (n & 1) : vec_at + M * E + sg * MH;
        };
        pn.add(fx, 1.f, at);
        p1.add(fx, -1.f, at);
        p0.add(fx, 1.f, at);
    }
    Pieces far[KEYMAJOR ? 2 * KS : 1];
    floatx4 acc2[2][4];                                                             // [sign][outer block], rows = features
    uint16_t* fw = Xi + w * 32 * LD;                                                // key-major: one piece of the wave's far rows, [sign, 16 features][E]
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
#pragma unroll
        for (int ob = 0; ob < 4; ++ob) acc2[sg][ob] = Frag<float>::zero();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const Pieces fp = split<3>(fx[sg * (2 * KS + 1) + 2 * ks], fx[sg * (2 * KS + 1) + 2 * ks + 1]);
            if (KEYMAJOR) far[KEYMAJOR ? sg * KS + ks : 0] = fp;
#pragma unroll
            for (int ob = 0; ob < 4; ++ob)
                acc2[sg][ob] = mma_pieces(fp, *reinterpret_cast<const uintx4*>(Yo + (16 * ob + r16) * LD + 32 * ks + 8 * g), acc2[sg][ob]);
        }
#pragma unroll
        for (int ob = 0; ob < 4; ++ob) acc2[sg][ob] -= fx[sg * (2 * KS + 1) + 2 * KS] * (KEYMAJOR ? 1.0f : co[16 * ob + r16]);
    }
    floatx4 acc3[KEYMAJOR ? EB : 1][KEYMAJOR ? 4 : 1];                              // d v: rows = value dims, columns = keys
    if (KEYMAJOR) {
#pragma unroll
        for (int eb = 0; eb < EB; ++eb)
#pragma unroll
            for (int ob = 0; ob < 4; ++ob) acc3[KEYMAJOR ? eb : 0][KEYMAJOR ? ob : 0] = Frag<float>::zero();
#pragma unroll
        for (int pc = 2; pc >= 0; --pc) {                                           // (small terms first)
#pragma unroll
            for (int n = 0; n < 2 * KS; ++n)
                *reinterpret_cast<uintx4*>(fw + (16 * (n / KS) + r16) * LD + 32 * (n % KS) + 8 * g) = far[KEYMAJOR ? n : 0].p[pc];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                      // (read by other lanes of the wave only)
            __builtin_amdgcn_wave_barrier();
            uintx4 tp[EB];
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) {
                const uint16_t* q = fw + (4 * g + (r16 >> 2)) * LD + 16 * eb + 4 * (r16 & 3);
                tp[eb] = lds_read_tr8(reinterpret_cast<const char*>(q), reinterpret_cast<const char*>(q + 16 * LD));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int ob = 0; ob < 4; ++ob) {
                const PiecesOf<NF> f = own_pieces(ob);
#pragma unroll
                for (int eb = 0; eb < EB; ++eb) {
                    floatx4& d = acc3[KEYMAJOR ? eb : 0][KEYMAJOR ? ob : 0];
#pragma unroll
                    for (int pf = NF - 1; pf >= 0; --pf)
                        if (pc + pf <= 2) d = mma_bf16(tp[eb], f.p[pf], d);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();                                                            // the far rows lie where the inner chunk goes
    }

    while (ic < c1) {
        const int n0 = ic * FC;
        if (!AHEAD) t.fetch(a, KEYMAJOR, xip, xis, yip, yis, bh, n0, len_i, base, kappa, tid);
        t.stash(a, Xi, Yi, diagi, exti, ci, tid);
        int nx = ic + 1;
        if (nx == e0) nx = max(nx, e1);                                             // (over the chunks inside the band)
        if (AHEAD && nx < c1) t.fetch(a, KEYMAJOR, xip, xis, yip, yis, bh, nx * FC, len_i, base, kappa, tid);
        __syncthreads();
        // (uniform) do the pairs of inner rows 32 st .. + 31 and outer rows 16 ob .. + 15 all lie in the band: a quarter of a chunk at a
        // window that is a multiple of 128, half on average otherwise.  (16 heads of 16384 tokens, window 1024, 256 features, training step:
        // 2108 -> 2071 us without their products)
        auto band_only = [&](int st, int ob) __attribute__((always_inline)) {
            const int rel = n0 + 32 * st - (o0 + 16 * ob);
            return rel - 15 >= -A && rel + 31 < Bq;
        };
        // df = g.v - c on the pairs outside the band, 0 inside: inner rows 32 st + 16 hb + 4 g + i, outer row 16 ob + r16 --
        // eight contraction slots of the products below -- in pieces
        for (int it = w; it < 8; it += NW) {
            const int st = it >> 2, ob = it & 3;
            if (band_only(st, ob)) continue;
            floatx4 s[2] = {Frag<float>::zero(), Frag<float>::zero()};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uintx4 yo = *reinterpret_cast<const uintx4*>(Yo + (16 * ob + r16) * LD + 32 * ks + 8 * g);
#pragma unroll
                for (int hb = 0; hb < 2; ++hb)
                    s[hb] = mma_bf16(*reinterpret_cast<const uintx4*>(Yi + (32 * st + 16 * hb + r16) * LD + 32 * ks + 8 * g), yo, s[hb]);
            }
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                const int row = 32 * st + 16 * hb + 4 * g;
                const floatx4 cq = *reinterpret_cast<const floatx4*>(ci + row);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int rel = n0 + row + i - (o0 + 16 * ob + r16);
                    s[hb][i] = (unsigned)(rel + A) < (unsigned)(A + Bq) ? 0.f : s[hb][i] - (KEYMAJOR ? cq[i] : co[16 * ob + r16]);
                }
            }
            const Pieces df = split<3>(s[0], s[1]);
#pragma unroll
            for (int pc = 0; pc < 3; ++pc) DF[(8 * pc + it) * 64 + lane] = df.p[pc];
        }
        __syncthreads();
        // acc2^T[feature][outer] += F^T[feature][inner] df[inner][outer]
        const bool fvalid = 16 * w + r16 < a.mh_valid;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            floatx4 f0[2], f1[2];
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                const int kb = 2 * st + hb;
                const floatx4 dd = P.rows_by_features(Xi + (16 * kb + r16) * LD + 8 * g);
                const floatx4 bias = *reinterpret_cast<const floatx4*>(exti + 16 * kb + 4 * g) - *reinterpret_cast<const floatx4*>(diagi + 16 * kb + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    f0[hb][i] = fvalid ? __builtin_amdgcn_exp2f(bias[i] + dd[i]) : 0.f;
                    f1[hb][i] = fvalid ? __builtin_amdgcn_exp2f(bias[i] - dd[i]) : 0.f;
                }
            }
            const PiecesOf<NF> fp[2] = {split<NF>(f0[0], f0[1]), split<NF>(f1[0], f1[1])};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ob = 0; ob < 4; ++ob) {
                if (band_only(st, ob)) continue;
                const Pieces df = {{DF[(4 * st + ob) * 64 + lane], DF[(8 + 4 * st + ob) * 64 + lane], DF[(16 + 4 * st + ob) * 64 + lane]}};
#pragma unroll
                for (int sg = 0; sg < 2; ++sg) acc2[sg][ob] = mma_pieces(fp[sg], df, acc2[sg][ob]);
            }
            if (KEYMAJOR) {
                // this wave's features of the low-rank weights outside the band: result rows = queries, columns = keys; then
                // d v^T[d][key] += g^T[d][query] W[query][key].  The operand is the one above transposed, one piece at a time
                // through the wave's rows in LDS
                PiecesOf<NF> wp[2];
#pragma unroll
                for (int pc = 0; pc < NF; ++pc) {
#pragma unroll
                    for (int sg = 0; sg < 2; ++sg) {
                        const uintx4 f = fp[sg].p[pc];
#pragma unroll
                        for (int hb = 0; hb < 2; ++hb)
                            *reinterpret_cast<uint2*>(ft + (16 * sg + r16) * FAR_LDT + 16 * hb + 4 * g) = make_uint2(f[2 * hb], f[2 * hb + 1]);
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");              // (read by other lanes of the wave only)
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb) {
                        const uint16_t* q = ft + (4 * g + (r16 >> 2)) * FAR_LDT + 16 * hb + 4 * (r16 & 3);
                        wp[hb].p[pc] = lds_read_tr8(reinterpret_cast<const char*>(q), reinterpret_cast<const char*>(q + 16 * FAR_LDT));
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_wave_barrier();
                }
                __builtin_amdgcn_sched_barrier(0);          // (the steps' operands do not fit the registers side by side)
#pragma unroll
                for (int ob = 0; ob < 4; ++ob) {
                    if (band_only(st, ob)) continue;
                    floatx4 wt[2];
                    const PiecesOf<NF> own = own_pieces(ob);
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb) {
                        wt[hb] = mma_pieces(wp[hb], own, Frag<float>::zero());
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int rel = n0 + 32 * st + 16 * hb + 4 * g + i - (o0 + 16 * ob + r16);
                            if ((unsigned)(rel + A) < (unsigned)(A + Bq)) wt[hb][i] = 0.f;
                        }
                    }
                    const Pieces wpc = split<3>(wt[0], wt[1]);
#pragma unroll
                    for (int eb = 0; eb < EB; ++eb) {
                        const uint16_t* yq = Yi + (32 * st + 4 * g + (r16 >> 2)) * LD + 16 * eb + 4 * (r16 & 3);
                        const uintx4 yt = lds_read_tr8(reinterpret_cast<const char*>(yq), reinterpret_cast<const char*>(yq + 16 * LD));
                        floatx4& d = acc3[KEYMAJOR ? eb : 0][KEYMAJOR ? ob : 0];
                        d = mma_pieces(yt, wpc, d);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();                                                            // the inner chunk and df are free
        ic = nx;
    }

    // the wave's rows of sqrt(t) P, asked for before the barriers of the reduction
    floatx4 pv[EB];
    const float stemp = sqrtf(a.temp);
#pragma unroll
    for (int eb = 0; eb < EB; ++eb)
#pragma unroll
        for (int i = 0; i < 4; ++i) pv[eb][i] = a.proj[(long)(16 * w + 4 * g + i) * E + 16 * eb + r16] * stemp;
    // u = F_o o acc2; d x = sqrt(t) P^T (u+ - u-) - t x sum u
    floatx4 du[4];
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) {
        floatx4 f0, f1;
        if (KEYMAJOR) {
            const PiecesOf<NF> x = own_pieces(ob);
            auto slot = [](uint32_t w, int odd) __attribute__((always_inline)) { return __uint_as_float(odd ? w & 0xffff0000u : w << 16); };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = i >> 1, odd = i & 1;
                f0[i] = slot(x.p[NF - 1][n], odd);
                f1[i] = slot(x.p[NF - 1][2 + n], odd);
#pragma unroll
                for (int pc = NF - 2; pc >= 0; --pc) {                               // (exact)
                    f0[i] += slot(x.p[pc][n], odd);
                    f1[i] += slot(x.p[pc][2 + n], odd);
                }
            }
        } else own_features(ob, f0, f1);
        const floatx4 up = f0 * acc2[0][ob], un = f1 * acc2[1][ob];
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s += up[i] + un[i];
        s = group_sum(s);
        if (g == 0) us[w * FC + 16 * ob + r16] = s;
        du[ob] = up - un;
    }
    // the wave's 16 rows of P as one 32-slot step: slots (0, 4 g + i) and (1, 4 g + i) carry different piece products
    uintx4 bo[4][3];
#pragma unroll
    for (int ob = 0; ob < 4; ++ob) {
        uint2 dh, dm, dl;
        split3_4(du[ob], dh, dm, dl);
        bo[ob][0] = uintx4{dh.x, dh.y, dh.x, dh.y};
        bo[ob][1] = uintx4{dm.x, dm.y, dm.x, dm.y};
        bo[ob][2] = uintx4{dl.x, dl.y, dh.x, dh.y};
    }
    constexpr int RC = far_reduce_cols<M, KEYMAJOR>(), RB = RC / 16;             // columns and 16-column blocks at a time
    constexpr int QUADS = FC * RC / 4;                                              // groups of four columns, per 64 rows
#pragma unroll
    for (int pass = 0; pass < (KEYMAJOR ? 2 : 1); ++pass)
#pragma unroll
        for (int e2 = 0; e2 < EB / RB; ++e2) {
#pragma unroll
          for (int eh = 0; eh < RB; ++eh) {
            const int eb = RB * e2 + eh;
            floatx4 d[4];
            if (pass == 0) {
                uint2 ph, pm, pl;
                split3_4(pv[eb], ph, pm, pl);
                const uintx4 a0 = {ph.x, ph.y, pm.x, pm.y}, a1 = {ph.x, ph.y, pl.x, pl.y};
#pragma unroll
                for (int ob = 0; ob < 4; ++ob) d[ob] = mma_bf16(a0, bo[ob][0], mma_bf16(a0, bo[ob][1], mma_bf16(a1, bo[ob][2], Frag<float>::zero())));
            } else {
#pragma unroll
                for (int ob = 0; ob < 4; ++ob) d[ob] = acc3[KEYMAJOR ? eb : 0][KEYMAJOR ? ob : 0];
            }
#pragma unroll
            for (int ob = 0; ob < 4; ++ob) *reinterpret_cast<floatx4*>(red + ((eh * NW + w) * FC + 16 * ob + r16) * 16 + 4 * g) = d[ob];
          }
            __syncthreads();
            float* dst = pass == 0 ? (KEYMAJOR ? a.dk : a.dq) : a.dv;
            for (int x = tid; x < QUADS; x += NT) {
                const int row = (x >> 2) % FC, qd = x & 3, eh = x / (4 * FC), eb = RB * e2 + eh;
                const float* rp = red + (eh * NW * FC + row) * 16 + 4 * qd;
                floatx4 s = *reinterpret_cast<const floatx4*>(rp);
                float usum = us[row];
#pragma unroll
                for (int v = 1; v < NW; ++v) {
                    s += *reinterpret_cast<const floatx4*>(rp + v * FC * 16);
                    usum += us[v * FC + row];
                }
                if (pass == 0) {
                    const uint2 xr = *reinterpret_cast<const uint2*>(Xo + row * LD + 16 * eb + 4 * qd);
                    const floatx4 xf = {__uint_as_float(xr.x << 16), __uint_as_float(xr.x & 0xffff0000u),
                                        __uint_as_float(xr.y << 16), __uint_as_float(xr.y & 0xffff0000u)};
                    s -= xf * (a.temp * usum);
                }
                if (o0 + row < Lo) *reinterpret_cast<floatx4*>(dst + ((long)bh * Lo + o0 + row) * E + 16 * eb + 4 * qd) = s;
            }
            __syncthreads();
        }
}

template <int E, int M, bool KEYMAJOR>
static int launch_lowrank(const FarArgs& a, hipStream_t st) {
    auto kern = far_lowrank_kernel<E, M, KEYMAJOR>;
    constexpr size_t smem = far_lowrank_smem<E, M, KEYMAJOR>();
    static std::atomic<unsigned long long> lds_set{0};     // (devices on which this kernel has its LDS limit)
    if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "far_lowrank")) return rc;
    const long items = (long)a.B * a.H * (KEYMAJOR ? a.n_kc : a.n_qc);
    const long grid = (items + a.n_xcd - 1) / a.n_xcd * a.n_xcd;
    if (grid > 2147483647L) return fail(ERR_ARG, "sblocal_bwd_far: too many workgroups");
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(2 * M), smem, st, a);
    return check_launch("far_lowrank_kernel");
}

template <int E, int M>
static int launch_far(const FarArgs& a, const LocalBwdArgs& band, hipStream_t st) {
    const int BH = a.B * a.H, per4 = M * (E + 1) / 4;
    const int k_segs = (a.n_kc + a.seg - 1) / a.seg, q_segs = (a.n_qc + a.seg - 1) / a.seg;
    hipLaunchKernelGGL((far_chunk_kernel<E, M>), dim3(k_segs + q_segs, BH), dim3(2 * M), 0, st, a);
    if (int rc = check_launch("far_chunk_kernel")) return rc;
    hipLaunchKernelGGL(far_scan_kernel, dim3((per4 + FAR_SCAN_NT - 1) / FAR_SCAN_NT, 2, BH), dim3(FAR_SCAN_NT), 0, st, a, per4);
    if (int rc = check_launch("far_scan_kernel")) return rc;
    if (int rc = launch_lowrank<E, M, false>(a, st)) return rc;
    if (int rc = launch_lowrank<E, M, true>(a, st)) return rc;
    return launch_local_bwd_exact(band, E, st);
}

// floats of each piece of the workspace, in order: c, kscale, qscale, kv, qg, dq, dk, dv
static void far_pieces(int64_t BH, int64_t T, int64_t S, int64_t E, int64_t M, int64_t (&n)[8]) {
    const int64_t kc = (S + FC - 1) / FC, qc = (T + FC - 1) / FC, per = M * (E + 1);
    const int64_t want[8] = {BH * T, BH * kc, BH * qc, BH * kc * per, BH * qc * per, BH * T * E, BH * S * E, BH * S * E};
    for (int i = 0; i < 8; ++i) n[i] = (want[i] + 63) / 64 * 64;
}

// chunks per segment: as many as leave 16 waves per compute unit (the chunk kernel holds 8), at most 16: the scan takes 227 us
// at one chunk per segment (16 heads of 16384 tokens, 256 features: it moves 1.1 GB), 54 us at 4, 30 at 8, 19 at 16, the
// chunk kernel the same at each
constexpr int FAR_MAX_SEG = 16;
static int far_segment(long BH, int n_kc, int n_qc, int M, int cus) {
    int seg = FAR_MAX_SEG;
    while (seg > 1 && BH * ((n_kc + seg - 1) / seg + (n_qc + seg - 1) / seg) * (M / 32) < 16L * cus) seg /= 2;
    return seg;
}

}  // namespace flyhip

using namespace flyhip;

extern "C" int64_t flyhip_sblocal_bwd_far_floats(int BH, int T, int S, int E, int M) {
    if (BH <= 0 || T <= 0 || S <= 0 || E <= 0 || M <= 0) return -1;
    int64_t n[8], sum = 0;
    far_pieces(BH, T, S, E, M, n);
    for (int64_t x : n) sum += x;
    return sum;
}

extern "C" int flyhip_sblocal_bwd_far(const void* q, const void* k, const void* v, const void* out, const void* grad_out,
                                      const float* log_norm, const float* proj, const int64_t* key_lengths,
                                      void* dq, void* dk, void* dv, float* workspace, int64_t workspace_floats,
                                      int B, int H, int T, int S, int E, int M, int mh_valid, int local_context,
                                      int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t k_sb, int64_t k_sh, int64_t k_ss,
                                      int64_t v_sb, int64_t v_sh, int64_t v_ss, int64_t o_sb, int64_t o_sh, int64_t o_ss,
                                      int64_t g_sb, int64_t g_sh, int64_t g_ss,
                                      int64_t dq_sb, int64_t dq_sh, int64_t dq_ss, int64_t dk_sb, int64_t dk_sh, int64_t dk_ss,
                                      int64_t dv_sb, int64_t dv_sh, int64_t dv_ss,
                                      float softmax_temp, void* stream) {
    FLY_REQUIRE(q && k && v && out && grad_out && log_norm && proj && dq && dk && dv && workspace, "sblocal_bwd_far: null pointer");
    FLY_REQUIRE(B > 0 && H > 0 && T > 0 && S > 0 && (int64_t)B * H <= 65535, "sblocal_bwd_far: empty problem or more than 65535 (batch, head) pairs");
    FLY_REQUIRE(local_context >= 1, "sblocal_bwd_far: local_context must be >= 1");
    FLY_REQUIRE(softmax_temp > 0.f, "sblocal_bwd_far: softmax_temp must be positive");
    FLY_REQUIRE(mh_valid >= 1 && 2 * mh_valid <= M, "sblocal_bwd_far: %d projection rows do not fit %d features", mh_valid, M);
    FLY_REQUIRE(((q_sb | q_sh | q_ss | k_sb | k_sh | k_ss | v_sb | v_sh | v_ss | g_sb | g_sh | g_ss | o_sb | o_sh | o_ss) % 8) == 0,
                "sblocal_bwd_far: input strides must be multiples of 8 elements (16-byte loads)");
    FLY_REQUIRE(((dq_sb | dq_sh | dq_ss | dk_sb | dk_sh | dk_ss | dv_sb | dv_sh | dv_ss) % 4) == 0,
                "sblocal_bwd_far: output strides must be multiples of 4 elements (8-byte stores)");
    FLY_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                  reinterpret_cast<uintptr_t>(grad_out) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(proj) |
                  reinterpret_cast<uintptr_t>(workspace)) % 16) == 0 &&
                ((reinterpret_cast<uintptr_t>(dq) | reinterpret_cast<uintptr_t>(dk) | reinterpret_cast<uintptr_t>(dv)) % 8) == 0,
                "sblocal_bwd_far: pointers must be 16-byte (inputs) and 8-byte (outputs) aligned");
    const int64_t need = flyhip_sblocal_bwd_far_floats(B * H, T, S, E, M);
    FLY_REQUIRE(workspace_floats >= need, "sblocal_bwd_far: workspace of %lld floats, %lld needed", (long long)workspace_floats, (long long)need);
    int64_t n[8];
    far_pieces((int64_t)B * H, T, S, E, M, n);
    float* p[8];
    float* at = workspace;
    for (int i = 0; i < 8; ++i) { p[i] = at; at += n[i]; }
    FarArgs a{reinterpret_cast<const uint16_t*>(q), reinterpret_cast<const uint16_t*>(k), reinterpret_cast<const uint16_t*>(v),
              reinterpret_cast<const uint16_t*>(grad_out), reinterpret_cast<const uint16_t*>(out), log_norm, proj, key_lengths,
              p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7],
              B, H, T, S, local_context, mh_valid, (S + FC - 1) / FC, (T + FC - 1) / FC,
              far_segment(B * H, (S + FC - 1) / FC, (T + FC - 1) / FC, M, machine().cus), q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, g_sb, g_sh, g_ss, o_sb, o_sh, o_ss, softmax_temp, machine().xcds};
    LocalBwdArgs band{q, k, v, grad_out, out, log_norm, p[0], key_lengths, dq, dk, dv, B, H, T, S, local_context,
                      q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, g_sb, g_sh, g_ss, o_sb, o_sh, o_ss,
                      dq_sb, dq_sh, dq_ss, dk_sb, dk_sh, dk_ss, dv_sb, dv_sh, dv_ss, softmax_temp, 0, p[5], p[6], p[7]};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    if (E == 32 && M == 32) return launch_far<32, 32>(a, band, st);
    if (E == 32 && M == 64) return launch_far<32, 64>(a, band, st);
    if (E == 64 && M == 32) return launch_far<64, 32>(a, band, st);
    if (E == 64 && M == 64) return launch_far<64, 64>(a, band, st);
    if (E == 64 && M == 128) return launch_far<64, 128>(a, band, st);
    if (E == 64 && M == 256) return launch_far<64, 256>(a, band, st);
    return fail(ERR_UNSUPPORTED, "sblocal_bwd_far: (head dim, features) = (%d, %d) not in "
                                 "{(32,32), (32,64), (64,32), (64,64), (64,128), (64,256)}", E, M);
}
