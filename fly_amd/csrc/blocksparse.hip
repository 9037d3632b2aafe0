// Block-sparse matmuls (SDD / DSD / DDS) and block-sparse row operations for gfx950.
//
// Sparse tensors are (Z, nnz, blk, blk) with block n the n-th nonzero of the (H, rows, cols)
// layout in row-major order.  Every matmul wave owns one register tile of the output (up to
// 32x32, built from 16x16 MFMA results) and walks its reduction list, reading operand fragments
// straight from global memory (16-byte / 8-byte vector loads when the contraction index is
// contiguous, strided gathers otherwise).  Products are formed with the operand that supplies
// the output columns on the MFMA "A" side, so a lane ends up with four consecutive output
// columns of one row and writes them with a single vector store.
#include "common.h"
#include <type_traits>
#include <math.h>

namespace flyhip {

template <typename T>
__device__ __forceinline__ typename Frag<T>::type frag_at(const T* p, long k_stride) {
    // four contraction elements starting at p, spaced by k_stride
    if (k_stride == 1) return Frag<T>::load(p);
    return Frag<T>::gather(p, k_stride);
}

template <typename T>
__device__ __forceinline__ void store_tile_row(T* p, long col_stride, floatx4 v, int ncols_left) {
    // v holds four consecutive output columns starting at p
    if (col_stride == 1 && ncols_left >= 4) { store4_f32(p, v); return; }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < ncols_left) p[i * col_stride] = Elem<T>::from_f32(v[i]);
}

// ---------------------------------------------------------------------------------------
// SDD: sparse = dense x dense^T
// ---------------------------------------------------------------------------------------
struct SddArgs {
    const void* a; const void* b; void* c; const int32_t* lut;
    int nnz, K;
    long a_sz, a_sh, a_sm, a_sk, b_sz, b_sh, b_sn, b_sk;
};

template <typename T, int BLK>
__global__ __launch_bounds__(256) void bs_sdd_kernel(SddArgs a) {
    constexpr int TILE = BLK >= 32 ? 32 : 16, NTL = TILE / 16, SUB = BLK / TILE;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const long wid = (long)blockIdx.x * 4 + w;
    const int n = (int)(wid / (SUB * SUB)), sub = (int)(wid % (SUB * SUB));
    if (n >= a.nnz) return;
    const int z = blockIdx.y;
    const int head = a.lut[4 * n], bi = a.lut[4 * n + 1], bj = a.lut[4 * n + 2], id = a.lut[4 * n + 3];
    const int ml = (sub / SUB) * TILE, nl = (sub % SUB) * TILE;      // tile origin inside the block
    const T* ap = reinterpret_cast<const T*>(a.a) + z * a.a_sz + head * a.a_sh + (long)(bi * BLK + ml) * a.a_sm;
    const T* bp = reinterpret_cast<const T*>(a.b) + z * a.b_sz + head * a.b_sh + (long)(bj * BLK + nl) * a.b_sn;

    floatx4 acc[NTL][NTL];
#pragma unroll
    for (int tm = 0; tm < NTL; ++tm)
#pragma unroll
        for (int tn = 0; tn < NTL; ++tn) acc[tm][tn] = Frag<float>::zero();

    for (int kk = 0; kk < a.K; kk += 16) {
        typename Frag<T>::type fa[NTL], fb[NTL];
#pragma unroll
        for (int t = 0; t < NTL; ++t) {
            fa[t] = frag_at<T>(ap + (long)(16 * t + r16) * a.a_sm + (long)(kk + 4 * g) * a.a_sk, a.a_sk);
            fb[t] = frag_at<T>(bp + (long)(16 * t + r16) * a.b_sn + (long)(kk + 4 * g) * a.b_sk, a.b_sk);
        }
#pragma unroll
        for (int tm = 0; tm < NTL; ++tm)
#pragma unroll
            for (int tn = 0; tn < NTL; ++tn) acc[tm][tn] = Frag<T>::mma(fb[tn], fa[tm], acc[tm][tn]);
    }
    // lane holds C[m = 16tm + r16][n = 16tn + 4g + i]
    T* cp = reinterpret_cast<T*>(a.c) + ((long)z * a.nnz + id) * (BLK * BLK);
#pragma unroll
    for (int tm = 0; tm < NTL; ++tm)
#pragma unroll
        for (int tn = 0; tn < NTL; ++tn)
            store4_f32(cp + (ml + 16 * tm + r16) * BLK + nl + 16 * tn + 4 * g, acc[tm][tn]);
}

// Fast SDD for 32x32 blocks of a 2-byte type with contiguous contraction (K a multiple of 32, at
// most 128): one wave per (head, block-row).  The wave loads the A fragments of its block-row once
// (16-byte loads, kept in registers) and then produces the row's blocks one after the other: B fragments with 16-byte loads, 16x16x32 MFMAs, 8-byte stores of a 2 KiB block.
// The hardware hands consecutive workgroup ids to the XCDs in turn (n_xcd of them), and every XCD has an L2
// of its own.  unit_of() turns a 1-D workgroup id into (unit, position inside the unit) such
// that all `per_unit` workgroups of a unit -- one (batch, head) matrix, whose dense operand they
// all re-read -- run on one XCD, so that operand comes from HBM once instead of once per XCD.
__device__ __forceinline__ bool unit_of(unsigned id, int n_xcd, int per_unit, int n_units, int& unit, int& pos) {
    const unsigned xcd = id % (unsigned)n_xcd, slot = id / (unsigned)n_xcd;
    unit = (int)(slot / per_unit) * n_xcd + (int)xcd;
    pos = (int)(slot % per_unit);
    return unit < n_units;
}
static long unit_grid(long n_units, long per_unit) {
    const long x = machine().xcds;
    return (n_units + x - 1) / x * x * per_unit;
}

template <typename T> __device__ __forceinline__ uint32_t pack2(float lo, float hi);
template <> __device__ __forceinline__ uint32_t pack2<bf16_t>(float lo, float hi) { return pack_bf16x2(lo, hi); }
template <> __device__ __forceinline__ uint32_t pack2<f16_t>(float lo, float hi) {
    const _Float16 l = (_Float16)lo, h = (_Float16)hi;
    return (uint32_t)__builtin_bit_cast(uint16_t, l) | ((uint32_t)__builtin_bit_cast(uint16_t, h) << 16);
}
template <typename T> __device__ __forceinline__ floatx4 mma32(uintx4 a, uintx4 b, floatx4 c);
template <> __device__ __forceinline__ floatx4 mma32<bf16_t>(uintx4 a, uintx4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ floatx4 mma32<f16_t>(uintx4 a, uintx4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8_t, a), __builtin_bit_cast(halfx8_t, b), c, 0, 0, 0);
}

struct SddRowArgs {
    const void* a; const void* b; void* c;
    const int32_t* row_ptr; const int32_t* row_blk; const int32_t* row_col;
    int nnz, K, brows_per_head, n_heads, Z;
    long a_sz, a_sh, a_sm, b_sz, b_sh, b_sn;
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
};

constexpr int SDD_RING = 3;

template <typename T, int KS>     // KS = K / 32
__global__ __launch_bounds__(256) void bs_sdd32_kernel(const SddRowArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    // one block-row per wave: the four waves of a workgroup walk neighbouring block-rows, whose
    // column lists mostly coincide, so their B-tile loads meet in the L1 cache
    int unit, grp;
    if (!unit_of(blockIdx.x, a.n_xcd, (a.brows_per_head + 3) / 4, a.n_heads * a.Z, unit, grp)) return;
    const int z = unit / a.n_heads, head = unit % a.n_heads, bi = grp * 4 + w;
    if (bi >= a.brows_per_head) return;
    const int brow = head * a.brows_per_head + bi;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const T* ap = reinterpret_cast<const T*>(a.a) + z * a.a_sz + head * a.a_sh + (long)(bi * 32 + r16) * a.a_sm + 8 * g;
    // MFMA row i of B-tile tn is block column 8*(i/4) + 4*tn + i%4: the four results a lane gets from
    // tile 0 and the four from tile 1 are then eight consecutive columns -> one 16-byte store
    const T* bp = reinterpret_cast<const T*>(a.b) + z * a.b_sz + head * a.b_sh +
                  (long)(8 * (r16 >> 2) + (r16 & 3)) * a.b_sn + 8 * g;
    T* cz = reinterpret_cast<T*>(a.c) + (long)z * a.nnz * 1024;
    if (nb == 0) return;
    uint4 fa[2][KS];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fa[tm][ks] = *reinterpret_cast<const uint4*>(ap + 16 * tm * a.a_sm + 32 * ks);
    // B tiles travel through a ring of SDD_RING register sets: the loads of block j + SDD_RING - 1
    // are issued before block j is multiplied and stored, so a wave keeps several tiles in flight
    uint4 fb[SDD_RING][2][KS];
    auto fetch = [&](uint4 (&dst)[2][KS], int j) {
        const long brow_b = (long)a.row_col[p0 + min(j, nb - 1)] * 32;
#pragma unroll
        for (int tn = 0; tn < 2; ++tn)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                dst[tn][ks] = *reinterpret_cast<const uint4*>(bp + (brow_b + 4 * tn) * a.b_sn + 32 * ks);
    };
#pragma unroll
    for (int u = 0; u < SDD_RING - 1; ++u) fetch(fb[u], u);
    for (int j0 = 0; j0 < nb; j0 += SDD_RING) {
#pragma unroll
        for (int u = 0; u < SDD_RING; ++u) {
            const int j = j0 + u;
            if (j >= nb) break;
            fetch(fb[(u + SDD_RING - 1) % SDD_RING], j + SDD_RING - 1);
            floatx4 acc[2][2];
#pragma unroll
            for (int tm = 0; tm < 2; ++tm)
#pragma unroll
                for (int tn = 0; tn < 2; ++tn) {
                    acc[tm][tn] = Frag<float>::zero();
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) acc[tm][tn] = Frag32<T>::mma(fb[u][tn][ks], fa[tm][ks], acc[tm][tn]);
                }
            // lane holds C[m = 16tm + r16][n = 8g + 4tn + i]: rows of 64 bytes, 16 consecutive rows per store
            T* cp = cz + (long)a.row_blk[p0 + j] * 1024;
#pragma unroll
            for (int tm = 0; tm < 2; ++tm) store8_f32(cp + (16 * tm + r16) * 32 + 8 * g, acc[tm][0], acc[tm][1]);
        }
    }
}

// Operand of a 16x16x32 MFMA whose contraction index runs down the rows of a row-major LDS tile
// ([k][feature]): lane (r16, g) needs feature f0 + r16 at k = 8g .. 8g + 7.  ds_read_b64_tr_b16 hands a lane
// the element column of a 16-lane group's 16 x 4 block of 2-byte values: with lane j of the group
// pointing at some row (its choice) for k-slot j / 4, columns 4 (j % 4) .. + 3, lane j receives column j of the
// four rows.  Two such reads (k-slots 8g .. 8g + 3 and 8g + 4 .. 8g + 7) make the eight k-slots; row_lo /
// row_hi are the LDS rows that hold k = 8g + r16 / 4 and k = 8g + 4 + r16 / 4 (tiles may keep their rows
// in any order).
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef unsigned int uintx2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uintx4 frag_down_rows_at(const uint16_t* tile, int ld, int f0, int r16, int row_lo, int row_hi) {
    typedef __attribute__((address_space(3))) shortx4 lds_shortx4;
    const uint16_t* p = tile + f0 + 4 * (r16 & 3);
    const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(p + row_lo * ld));
    const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(p + row_hi * ld));
    const uintx2 l = __builtin_bit_cast(uintx2, lo), h = __builtin_bit_cast(uintx2, hi);
    return uintx4{l[0], l[1], h[0], h[1]};
}

// SDD for layouts whose neighbouring block-rows share most of their columns (band and butterfly
// patterns do): one workgroup per (batch, head, four consecutive block-rows), wave w owning row
// 4*group + w with its A fragments in registers.  The workgroup walks the union of the four
// column lists (uni_inner), stages each 32 x K tile of B once in LDS -- a quarter of the cache
// traffic of the one-wave-per-row kernel -- and every wave whose row holds that column
// (uni_blk[step][w] >= 0) multiplies and stores its 2 KiB block.  Tiles are double-buffered:
// the global loads of step s+1 are in flight while step s is multiplied.
struct SddUniArgs {
    const void* a; const void* b; void* c;
    const int32_t* uni_ptr; const int32_t* uni_inner; const int32_t* uni_blk;
    int nnz, brows_per_head, grps_per_head, n_heads, Z;
    long a_sz, a_sh, a_sm, b_sz, b_sh, b_sn;
    // EPI 1: c = scale * p * (a b^T - delta[row]) on the nonzero blocks, the gradient of the scores of a
    // softmax(scale * s) -> p -> p v chain from a = d out, b = v, delta = rowsum(d out * out)
    // EPI 2: c = 2^(scale * a b^T - delta[row]): the probabilities again from a = q, b = k, scale =
    // softmax scale * log2(e) and delta = the rows' base-2 log-denominators of the one-kernel attention
    const void* p; const float* delta; float scale;
    // EPI 3: both at once from a = d out, b = v and a2 = q, b2 = k (strides as a, b): p2 = 2^(scale2 * a2 b2^T -
    // lse2[row]) is written to p2 and c = scale * p2 * (a b^T - delta[row])
    const void* a2; const void* b2; const float* lse2; void* p2; float scale2;
    long a2_sz, a2_sh, a2_sm, b2_sz, b2_sh, b2_sn;
    // ... and the gradient of a2 on the way: dq = c b2 (rows of a2), accumulated over the row's blocks
    void* dq; long dq_sz, dq_sh, dq_sm;
    // ... with delta formed here when `out` is given (delta may then be null): rowsum(a * out), out laid out like a
    const void* out; long o_sz, o_sh, o_sm;
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
    // EPI 3 with DROP: the forward dropped probabilities by the hash of (seed, row = (z H + head) L + query, key)
    // (drop_keep): p2 is then written with the dropped ones zeroed and the kept ones scaled by 1 / (1 - p) -- the
    // operand of dV -- and c = scale * p * (m * (a b^T) - delta[row]) with m that 0 or 1 / (1 - p)
    uint32_t drop_seed, drop_thresh; float drop_scale;
};

template <typename T, int KS, int EPI = 0, bool DROP = false>     // KS = K / 32; EPI: 0 product, 1 softmax gradient, 2 probabilities
__global__ __launch_bounds__(256) void bs_sdd32u_kernel(const SddUniArgs a) {
    static_assert(!DROP || EPI == 3, "dropout belongs to the epilogue that forms the probabilities again");
    constexpr bool DSOFT = EPI == 1, PROB = EPI == 2, BOTH = EPI == 3;
    constexpr int K = 32 * KS, LD = K + 8;              // LDS row stride: 16 rows of a tile hit all banks once
    constexpr int CPR = K / 8;                          // 16-byte chunks per tile row
    constexpr int NCH = (32 * CPR + 255) / 256;         // chunks per thread
    __shared__ __attribute__((aligned(16))) uint16_t tile[2][32 * LD];
    __shared__ __attribute__((aligned(16))) uint16_t tile2[BOTH ? 2 : 1][BOTH ? 32 * LD : 8];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int unit, grp;
    if (!unit_of(blockIdx.x, a.n_xcd, a.grps_per_head, a.n_heads * a.Z, unit, grp)) return;
    const int z = unit / a.n_heads, head = unit % a.n_heads;
    const int ug = head * a.grps_per_head + grp;
    const int p0 = a.uni_ptr[ug], n = a.uni_ptr[ug + 1] - p0;
    const int bi = grp * 4 + w;
    const bool have_row = bi < a.brows_per_head;
    if (n == 0) {
        if (EPI == 3 && have_row) {                     // rows without blocks: zero gradient
            T* dqp = reinterpret_cast<T*>(a.dq) + z * a.dq_sz + head * a.dq_sh;
            for (int e = lane; e < 32 * K / 4; e += 64)
                store4_f32(dqp + (long)(bi * 32 + e / (K / 4)) * a.dq_sm + 4 * (e % (K / 4)), Frag<float>::zero());
        }
        return;
    }
    const T* ap = reinterpret_cast<const T*>(a.a) + z * a.a_sz + head * a.a_sh +
                  (long)(min(bi, a.brows_per_head - 1) * 32 + r16) * a.a_sm + 8 * g;
    const T* bz = reinterpret_cast<const T*>(a.b) + z * a.b_sz + head * a.b_sh;
    T* cz = reinterpret_cast<T*>(a.c) + (long)z * a.nnz * 1024;
    // DSOFT: this lane's rows are 16 tm + r16 of block-row bi
    const long rowvec_off = ((long)z * a.n_heads + head) * a.brows_per_head * 32 + (long)min(bi, a.brows_per_head - 1) * 32 + r16;
    const float* dlt = (DSOFT || PROB || (BOTH && a.delta)) ? a.delta + rowvec_off : nullptr;
    uintx4 fa[2][KS];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fa[tm][ks] = *reinterpret_cast<const uintx4*>(ap + 16 * tm * a.a_sm + 32 * ks);
    // EPI 3: the second product's row operand, column tiles and row vector
    uintx4 fa2[BOTH ? 2 : 1][BOTH ? KS : 1];
    const T* bz2 = nullptr;
    float lse_row[2] = {0.f, 0.f}, dl_row[2] = {0.f, 0.f};
    if (BOTH) {
        const T* ap2 = reinterpret_cast<const T*>(a.a2) + z * a.a2_sz + head * a.a2_sh +
                       (long)(min(bi, a.brows_per_head - 1) * 32 + r16) * a.a2_sm + 8 * g;
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) fa2[BOTH ? tm : 0][BOTH ? ks : 0] = *reinterpret_cast<const uintx4*>(ap2 + 16 * tm * a.a2_sm + 32 * ks);
            lse_row[tm] = a.lse2[rowvec_off + 16 * tm];
            if (a.out) {
                // delta = sum over the head dim of d out * out for this lane's row: the lane holds 8 KS of the
                // row's values, the four lanes r16 + 16g the rest
                const T* op = reinterpret_cast<const T*>(a.out) + z * a.o_sz + head * a.o_sh +
                              (long)(min(bi, a.brows_per_head - 1) * 32 + 16 * tm + r16) * a.o_sm + 8 * g;
                float part = 0.f;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const uintx4 ov = *reinterpret_cast<const uintx4*>(op + 32 * ks);
                    const uintx4 gv = fa[tm][ks];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        T x, y;
                        *reinterpret_cast<uint16_t*>(&x) = (uint16_t)(gv[e >> 1] >> (16 * (e & 1)));
                        *reinterpret_cast<uint16_t*>(&y) = (uint16_t)(ov[e >> 1] >> (16 * (e & 1)));
                        part += Elem<T>::to_f32(x) * Elem<T>::to_f32(y);
                    }
                }
                dl_row[tm] = group_sum(part);
            } else {
                dl_row[tm] = dlt[16 * tm];
            }
        }
        bz2 = reinterpret_cast<const T*>(a.b2) + z * a.b2_sz + head * a.b2_sh;
    }
    uint32_t drop_row[2] = {0u, 0u};
    if (DROP) {
        const uint32_t row0 = (uint32_t)rowvec_off;     // (z H + head) L + 32 bi + r16
        drop_row[0] = drop_row_hash(a.drop_seed, row0);
        drop_row[1] = drop_row_hash(a.drop_seed, row0 + 16u);
    }

    // staging: chunk c = tid + 256 i is 16 bytes of tile row c / CPR.  Block column n lands in LDS row
    // 16*((n>>2)&1) + 4*(n>>3) + (n&3), so that MFMA tile tn reads the 16 consecutive LDS rows
    // 16 tn .. 16 tn + 15 and its row i is block column 8*(i/4) + 4*tn + i%4: the four results a lane
    // gets from tile 0 and the four from tile 1 are eight consecutive columns -> one 16-byte store
    uintx4 reg[NCH], reg2[BOTH ? NCH : 1];
    auto fetch = [&](int inner) __attribute__((always_inline)) {
        const long brow_b = (long)inner * 32;
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = tid + 256 * i;
            if (c < 32 * CPR) reg[i] = *reinterpret_cast<const uintx4*>(bz + (brow_b + c / CPR) * a.b_sn + 8 * (c % CPR));
            if (BOTH && c < 32 * CPR)
                reg2[BOTH ? i : 0] = *reinterpret_cast<const uintx4*>(bz2 + (brow_b + c / CPR) * a.b2_sn + 8 * (c % CPR));
        }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = tid + 256 * i, nrow = c / CPR;
            const int lrow = 16 * ((nrow >> 2) & 1) + 4 * (nrow >> 3) + (nrow & 3);
            if (c < 32 * CPR) *reinterpret_cast<uintx4*>(&tile[buf][lrow * LD + 8 * (c % CPR)]) = reg[i];
            if (BOTH && c < 32 * CPR) *reinterpret_cast<uintx4*>(&tile2[BOTH ? buf : 0][lrow * LD + 8 * (c % CPR)]) = reg2[BOTH ? i : 0];
        }
    };
    floatx4 dqa[BOTH ? 2 * KS : 1][2];                  // dq^T[feature 16dt + 4g + i][row 16tm + r16]
    if (BOTH) {
#pragma unroll
        for (int dt = 0; dt < 2 * KS; ++dt) { dqa[BOTH ? dt : 0][0] = Frag<float>::zero(); dqa[BOTH ? dt : 0][1] = Frag<float>::zero(); }
    }
    // the index lists are read two steps (block-column) and one step (block id) ahead of their use
    int inner_n1 = n > 1 ? a.uni_inner[p0 + 1] : 0;
    int blk = a.uni_blk[(long)p0 * 4 + w];
    int inner_cur = a.uni_inner[p0];
    fetch(inner_cur);
    stash(0);
    drain_loads();
    __syncthreads();
    for (int s = 0; s < n; ++s) {
        const int inner_n2 = s + 2 < n ? a.uni_inner[p0 + s + 2] : 0;
        const int blk_n1 = s + 1 < n ? a.uni_blk[(long)(p0 + s + 1) * 4 + w] : -1;
        if (s + 1 < n) fetch(inner_n1);
        const bool mine = blk >= 0 && have_row;
        floatx4 acc[2][2], acc2[2][2];
        uintx4 pv[2];
        if (DSOFT && mine) {                              // requested before the products, used after them
            const T* pp = reinterpret_cast<const T*>(a.p) + ((long)z * a.nnz + blk) * 1024;
#pragma unroll
            for (int tm = 0; tm < 2; ++tm)
                pv[tm] = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(pp + (16 * tm + r16) * 32 + 8 * g));
        }
        if (mine) {
            const uint16_t* tp = tile[s & 1];
            uintx4 fb[2][KS];
#pragma unroll
            for (int tn = 0; tn < 2; ++tn)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    fb[tn][ks] = *reinterpret_cast<const uintx4*>(tp + (16 * tn + r16) * LD + 32 * ks + 8 * g);
#pragma unroll
            for (int tm = 0; tm < 2; ++tm)
#pragma unroll
                for (int tn = 0; tn < 2; ++tn) {
                    acc[tm][tn] = Frag<float>::zero();
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) acc[tm][tn] = mma32<T>(fb[tn][ks], fa[tm][ks], acc[tm][tn]);
                }
            if (BOTH) {
                const uint16_t* tp2 = tile2[BOTH ? (s & 1) : 0];
#pragma unroll
                for (int tn = 0; tn < 2; ++tn)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        fb[tn][ks] = *reinterpret_cast<const uintx4*>(tp2 + (16 * tn + r16) * LD + 32 * ks + 8 * g);
#pragma unroll
                for (int tm = 0; tm < 2; ++tm)
#pragma unroll
                    for (int tn = 0; tn < 2; ++tn) {
                        acc2[tm][tn] = Frag<float>::zero();
#pragma unroll
                        for (int ks = 0; ks < KS; ++ks)
                            acc2[tm][tn] = mma32<T>(fb[tn][ks], fa2[BOTH ? tm : 0][BOTH ? ks : 0], acc2[tm][tn]);
                    }
            }
        }
        // the next tile goes to LDS before this step's stores are issued: the wait for its loads would
        // otherwise wait for the stores too (one counter covers both)
        if (s + 1 < n) stash((s + 1) & 1);
        if (mine) {
            // lane holds C[m = 16tm + r16][n = 8g + 4tn + i]
            T* cp = cz + (long)blk * 1024;
#pragma unroll
            for (int tm = 0; tm < 2; ++tm) {
                if (DSOFT) {
                    const float dl = dlt[16 * tm];
#pragma unroll
                    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t word = pv[tm][2 * tn + (i >> 1)];
                            T e;
                            *reinterpret_cast<uint16_t*>(&e) = (i & 1) ? (uint16_t)(word >> 16) : (uint16_t)(word & 0xffffu);
                            acc[tm][tn][i] = a.scale * Elem<T>::to_f32(e) * (acc[tm][tn][i] - dl);
                        }
                }
                if (BOTH) {
#pragma unroll
                    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(acc2[tm][tn][i], a.scale2, -lse_row[tm]));
                            if (DROP) {
                                const uint32_t col = (uint32_t)inner_cur * 32u + 8u * g + 4u * tn + i;
                                const float m = drop_keep(drop_row[tm], col, a.drop_thresh) ? a.drop_scale : 0.f;
                                acc2[tm][tn][i] = m * pr;
                                acc[tm][tn][i] = a.scale * pr * (m * acc[tm][tn][i] - dl_row[tm]);
                            } else {
                                acc2[tm][tn][i] = pr;
                                acc[tm][tn][i] = a.scale * pr * (acc[tm][tn][i] - dl_row[tm]);
                            }
                        }
                    T* pp2 = reinterpret_cast<T*>(a.p2) + ((long)z * a.nnz + blk) * 1024;
                    store8_f32(pp2 + (16 * tm + r16) * 32 + 8 * g, acc2[tm][0], acc2[tm][1]);
                    // the lane's eight ds values are columns 8g .. 8g+7 of row 16tm + r16: an MFMA operand as they are
                    const uintx4 dsb = {pack2<T>(acc[tm][0][0], acc[tm][0][1]), pack2<T>(acc[tm][0][2], acc[tm][0][3]),
                                        pack2<T>(acc[tm][1][0], acc[tm][1][1]), pack2<T>(acc[tm][1][2], acc[tm][1][3])};
                    // ... against the b2 tile read down its rows (block column n sits in LDS row
                    // 16 ((n >> 2) & 1) + 4 (n >> 3) + (n & 3), see the staging)
                    const uint16_t* tt = tile2[BOTH ? (s & 1) : 0];
                    const int n_lo = 8 * g + (r16 >> 2), n_hi = n_lo + 4;
                    const int row_lo = 16 * ((n_lo >> 2) & 1) + 4 * (n_lo >> 3) + (n_lo & 3);
                    const int row_hi = 16 * ((n_hi >> 2) & 1) + 4 * (n_hi >> 3) + (n_hi & 3);
#pragma unroll
                    for (int dt = 0; dt < 2 * KS; ++dt) {
                        const uintx4 fk = frag_down_rows_at(tt, LD, 16 * dt, r16, row_lo, row_hi);
                        dqa[BOTH ? dt : 0][tm] = mma32<T>(fk, dsb, dqa[BOTH ? dt : 0][tm]);
                    }
                }
                if (PROB) {
                    const float dl = dlt[16 * tm];
#pragma unroll
                    for (int tn = 0; tn < 2; ++tn)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[tm][tn][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[tm][tn][i], a.scale, -dl));
                }
                store8_f32(cp + (16 * tm + r16) * 32 + 8 * g, acc[tm][0], acc[tm][1]);
            }
        }
        inner_cur = inner_n1;
        inner_n1 = inner_n2;
        blk = blk_n1;
        __syncthreads();
    }
    if (BOTH && have_row) {
        T* dqp = reinterpret_cast<T*>(a.dq) + z * a.dq_sz + head * a.dq_sh;
#pragma unroll
        for (int tm = 0; tm < 2; ++tm)
#pragma unroll
            for (int dt = 0; dt < 2 * KS; ++dt)
                store4_f32(dqp + (long)(bi * 32 + 16 * tm + r16) * a.dq_sm + 16 * dt + 4 * g, dqa[BOTH ? dt : 0][tm]);
    }
}

// ---------------------------------------------------------------------------------------
// SDD with the contraction index slowest in both operands: sparse = A^T B, A (K x M), B (K x N)
// ---------------------------------------------------------------------------------------
// The weight gradient of a block-sparse linear layer: K = tokens (tens of thousands), M / N = output / input features, 32x32
// blocks of a 2-byte type.  One workgroup of eight waves per (group of <= 4 consecutive block-rows with identical column
// lists, chunk of <= 2 NP of their block-columns, slice of K): a 128 x 64 NP output tile, wave (wm, wn) owning 64 rows and
// every fourth 16-column tile.  What bounds it is the operands' way into LDS: a 128 x 128 tile per workgroup reads the
// output gradient once for every four columns of a list (262 us for the widening layer of a channel MLP at 50176 tokens: 9
// columns in chunks of 4, 4 and 1), so a chunk takes up to ten.  Per step of 32 tokens the tiles go from memory straight
// into LDS, three steps ahead in four stages; the MFMA fragments, whose contraction index runs down the rows, are two
// transposing 8-byte LDS reads each.  A holds [token][128 features], B [pair of list entries][token][64 features] (both
// entries of a pair in one 128-byte line where they are neighbours), 32-byte pieces XOR-swizzled by the token so that the
// eight rows a half-wave reads together cover all banks.  Measured (us, before / now, with the zero fill and the rounding):
// 768 -> 3072 features 267 / 161, 3072 -> 768 229 / 188, 1024 -> 4096 343 / 243, 768 -> 768 124 / 70 at 50176 tokens; 104 / 55, 102 / 57, 139 / 63,
// 44 / 40 at 8192; 32 to 33 on either side at 512, where the host is the slower one.  The slices' partial blocks meet in an fp32 buffer through hardware
// float atomics (the caller zeroes it and rounds it to the output type afterwards).
struct SddKArgs {
    const void* a; const void* b; float* c32;
    const int32_t* seg_ptr; const int32_t* seg_blk; const int32_t* seg_inner;
    const int32_t* grp_row0; const int32_t* grp_n;
    int per_head, K, k_slice, chunks, nnz;
    long a_sz, a_sh, a_sk, b_sz, b_sh, b_sk;
    int n_grp, slices, n_xcd;
};
constexpr int SDDK_STAGES = 4, SDDK_MAX_PAIRS = 5;
constexpr int sddk_stage_bytes(int np) { return 8192 + 4096 * np; }

template <typename T, int NP>
__global__ __launch_bounds__(512) void bs_sdd32k_kernel(const SddKArgs a) {
    constexpr int NI = (8 + 4 * NP + 7) / 8;                // transfers of 1 KB a wave and step
    constexpr int STAGE = sddk_stage_bytes(NP);
    extern __shared__ __attribute__((aligned(128))) char sddk_smem[];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int wm = w & 1, wn = w >> 1, z = blockIdx.z;
    // (slice, group, chunk) dealt to the dies in contiguous runs: the groups that read one slice of the inputs share an L2
    const int n_items = a.n_grp * a.chunks * a.slices, per_xcd = (n_items + a.n_xcd - 1) / a.n_xcd;
    const int item = (blockIdx.x % a.n_xcd) * per_xcd + blockIdx.x / a.n_xcd;
    if (blockIdx.x / a.n_xcd >= per_xcd || item >= n_items) return;             // workgroup-uniform
    const int chunk = item % a.chunks, grp = item / a.chunks % a.n_grp, slice = item / (a.chunks * a.n_grp);
    const int row0 = a.grp_row0[grp], gn = a.grp_n[grp];
    const int head = row0 / a.per_head, brow0 = row0 % a.per_head;
    const int p0 = a.seg_ptr[row0], nin = a.seg_ptr[row0 + 1] - p0;
    const int j0 = chunk * 2 * NP, jn = min(2 * NP, nin - j0);                  // this chunk's list entries j0 .. j0 + jn - 1
    const int k0 = slice * a.k_slice, k1 = min(a.K, k0 + a.k_slice);
    if (jn <= 0 || k0 >= k1) return;                                            // workgroup-uniform
    const char* ap = reinterpret_cast<const char*>(a.a) + 2 * (z * a.a_sz + head * a.a_sh + (long)brow0 * 32);
    const char* bp = reinterpret_cast<const char*>(a.b) + 2 * (z * a.b_sz + head * a.b_sh);

    // transfer w + 8 i of a step: 0..7 bring four tokens of A each, 8 + 4 r + j tokens 8 j .. 8 j + 7 of pair r of B (one past
    // the last is the wave's first again: every wave issues NI a step, which is what the waits count).  A lane's 16 bytes:
    // the token's bytes from `col` on; absent blocks are read from a present one and their products not stored
    const char* src[NI];
    long stride[NI];
    int tok[NI], dst[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int t = w + 8 * i < 8 + 4 * NP ? w + 8 * i : w;                   // (wave-uniform)
        if (t < 8) {
            const int tk = 4 * t + (lane >> 4), c = lane & 15;
            const int p = (c >> 1) ^ ((tk & 3) + 4 * ((tk >> 3) & 1));
            tok[i] = tk;
            src[i] = ap + (p < 2 * gn ? 32 * p : 32 * (p & 1)) + 16 * (c & 1);
            stride[i] = 2 * a.a_sk;
            dst[i] = 1024 * t;
        } else {
            const int r = (t - 8) >> 2, tk = 8 * ((t - 8) & 3) + (lane >> 3), c = lane & 7;
            const int p = (c >> 1) ^ (((tk >> 1) & 1) + 2 * ((tk >> 3) & 1));
            const int inner = a.seg_inner[p0 + j0 + min(2 * r + (p >> 1), jn - 1)];
            tok[i] = tk;
            src[i] = bp + (long)inner * 64 + 32 * (p & 1) + 16 * (c & 1);
            stride[i] = 2 * a.b_sk;
            dst[i] = 8192 + 4096 * r + 1024 * ((t - 8) & 3);
        }
    }
    auto transfer = [&](int kt, int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NI; ++i)                                            // (clamped; tokens past k1 are zeroed below)
            dma_to_lds(src[i] + min(kt + tok[i], a.K - 1) * stride[i], sddk_smem + stage * STAGE + dst[i]);
    };

    floatx4 acc[4][NP];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NP; ++j) acc[i][j] = Frag<float>::zero();
    const int trow = 8 * g + (r16 >> 2);                                        // (+ 4 for the second half: same swizzle)
    const int aoff = trow * 256 + 8 * (r16 & 3), asw = (trow & 3) + 4 * (g & 1);
    const int boff = 8192 + trow * 128 + 32 * (wn ^ (((trow >> 1) & 1) + 2 * (g & 1))) + 8 * (r16 & 3);
    auto compute = [&](const char* st, bool ragged, int left) __attribute__((always_inline)) {
        uintx4 keep = {~0u, ~0u, ~0u, ~0u};                                     // tokens 8 g .. 8 g + 7 of the step that exist
        if (ragged) {
#pragma unroll
            for (int d = 0; d < 4; ++d)
                keep[d] = (8 * g + 2 * d < left ? 0xffffu : 0u) | (8 * g + 2 * d + 1 < left ? 0xffff0000u : 0u);
        }
        uintx4 fa[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const char* q = st + aoff + 32 * ((4 * wm + i) ^ asw);
            fa[i] = lds_read_tr8(q, q + 4 * 256);
            if (ragged) fa[i] &= keep;
        }
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const char* q = st + boff + 4096 * j;
            uintx4 fb = lds_read_tr8(q, q + 4 * 128);
            if (ragged) fb &= keep;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][j] = mma32<T>(fa[i], fb, acc[i][j]);
        }
    };
#pragma unroll
    for (int d = 0; d < SDDK_STAGES - 1; ++d) transfer(k0 + 32 * d, d);
    int cur = 0;
    for (int kt = k0; kt < k1; kt += 32) {
        drain_loads_but<NI * (SDDK_STAGES - 2)>();                              // this wave's part of the step is in LDS
        __syncthreads();                                                        // everyone's is; the stage before it is free
        transfer(kt + 32 * (SDDK_STAGES - 1), (cur + SDDK_STAGES - 1) % SDDK_STAGES);
        if (kt + 32 <= k1) compute(sddk_smem + cur * STAGE, false, 32);
        else compute(sddk_smem + cur * STAGE, true, k1 - kt);
        cur = (cur + 1) % SDDK_STAGES;
    }
    drain_loads();                                                              // nothing may land in LDS after the workgroup has ended
    // lane holds C[out = 64 wm + 16 i + 4 g + x][in = 16 (wn + 4 j) + r16] of the chunk
    float* cz = a.c32 + (long)z * a.nnz * 1024;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int ob = 2 * wm + (i >> 1);
        if (ob >= gn) continue;
        const int* blks = a.seg_blk + a.seg_ptr[row0 + ob] + j0;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int t = wn + 4 * j;
            if (t >> 1 >= jn) continue;
            float* cb = cz + (long)blks[t >> 1] * 1024 + (16 * (i & 1) + 4 * g) * 32 + 16 * (t & 1) + r16;
#pragma unroll
            for (int x = 0; x < 4; ++x) unsafeAtomicAdd(cb + 32 * x, acc[i][j][x]);
        }
    }
}

// ---------------------------------------------------------------------------------------
// DSD: dense = sparse x dense
// ---------------------------------------------------------------------------------------
struct DxdArgs {
    const void* sp; const void* dn; void* c;
    const int32_t* seg_ptr; const int32_t* seg_blk; const int32_t* seg_inner;
    int n_seg, per_head, X, trans;      // X = N (DSD: dense columns) or M (DDS: dense rows)
    long sp_sz;
    long dn_sz, dn_sh, dn_s0, dn_s1;    // DSD: (k, n) strides; DDS: (m, k) strides
    long c_sz, c_sh, c_sm, c_sn;
    int Z;
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
    const void* bias;   // DDS, optional: one value per output column
};

template <typename T, int BLK>
__global__ __launch_bounds__(256) void bs_dsd_kernel(DxdArgs a) {
    constexpr int TILE = BLK >= 32 ? 32 : 16, NTL = TILE / 16, SUBM = BLK / TILE;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const int ntn = (a.X + 31) / 32;
    const long wid = (long)blockIdx.x * 4 + w;
    const long per_seg = (long)SUBM * ntn;
    const int seg = (int)(wid / per_seg);
    if (seg >= a.n_seg) return;
    const int rem = (int)(wid % per_seg), subm = rem / ntn, nt = rem % ntn;
    const int z = blockIdx.y;
    const int head = seg / a.per_head, brow = seg % a.per_head;
    const int n0 = nt * 32;
    const T* spz = reinterpret_cast<const T*>(a.sp) + z * a.sp_sz;
    const T* dnp = reinterpret_cast<const T*>(a.dn) + z * a.dn_sz + head * a.dn_sh;

    floatx4 acc[NTL][2];
#pragma unroll
    for (int tm = 0; tm < NTL; ++tm) { acc[tm][0] = Frag<float>::zero(); acc[tm][1] = Frag<float>::zero(); }
    bool nok[2];
    nok[0] = n0 + r16 < a.X;
    nok[1] = n0 + 16 + r16 < a.X;

    const int p1 = a.seg_ptr[seg + 1];
    for (int p = a.seg_ptr[seg]; p < p1; ++p) {
        const T* blkp = spz + (long)a.seg_blk[p] * (BLK * BLK);
        const long krow0 = (long)a.seg_inner[p] * BLK;
#pragma unroll
        for (int kk = 0; kk < BLK; kk += 16) {
            typename Frag<T>::type fs[NTL], fd[2];
#pragma unroll
            for (int tm = 0; tm < NTL; ++tm) {
                const int m = subm * TILE + 16 * tm + r16;
                fs[tm] = a.trans ? Frag<T>::gather(blkp + (kk + 4 * g) * BLK + m, BLK)
                                 : Frag<T>::load(blkp + m * BLK + kk + 4 * g);
            }
#pragma unroll
            for (int tn = 0; tn < 2; ++tn) {
                fd[tn] = Frag<T>::zero();
                if (nok[tn])
                    fd[tn] = frag_at<T>(dnp + (krow0 + kk + 4 * g) * a.dn_s0 + (long)(n0 + 16 * tn + r16) * a.dn_s1, a.dn_s0);
            }
#pragma unroll
            for (int tm = 0; tm < NTL; ++tm) {
                acc[tm][0] = Frag<T>::mma(fd[0], fs[tm], acc[tm][0]);
                acc[tm][1] = Frag<T>::mma(fd[1], fs[tm], acc[tm][1]);
            }
        }
    }
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh;
#pragma unroll
    for (int tm = 0; tm < NTL; ++tm) {
        const long m = (long)brow * BLK + subm * TILE + 16 * tm + r16;
#pragma unroll
        for (int tn = 0; tn < 2; ++tn) {
            const int n = n0 + 16 * tn + 4 * g;
            if (n < a.X) store_tile_row<T>(cp + m * a.c_sm + n * a.c_sn, a.c_sn, acc[tm][tn], a.X - n);
        }
    }
}

// Fast DSD for 32x32 blocks of a 2-byte type, dense operand with contiguous columns (the V of
// attention): one workgroup per (head, block-row, 64-column tile).  Wave w reduces the row's blocks
// w, w+4, ...: the sparse block supplies k-contiguous fragments straight from global memory; the
// 32 x 64 tile of the dense operand is staged in a wave-private LDS buffer (16-byte global loads)
// and read back column-wise, which is the transposition a [k][n] operand needs.  The four partial
// sums meet in LDS and leave as 16-byte stores.
constexpr int DSD_LD = 68;      // LDS row stride in elements: the four k-groups of a read hit distinct banks

template <typename T>
__global__ __launch_bounds__(256) void bs_dsd32_kernel(DxdArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t vt[4][32 * DSD_LD];
    __shared__ float part[4][32][64 + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, g = lane >> 4;
    const int ntn = (a.X + 63) / 64, n_heads = a.n_seg / a.per_head;
    int unit, pos;
    if (!unit_of(blockIdx.x, a.n_xcd, a.per_head * ntn, n_heads * a.Z, unit, pos)) return;
    const int z = unit / n_heads, head = unit % n_heads, brow = pos / ntn, n0 = (pos % ntn) * 64;
    const int seg = head * a.per_head + brow;
    const T* spz = reinterpret_cast<const T*>(a.sp) + z * a.sp_sz;
    const T* dnp = reinterpret_cast<const T*>(a.dn) + z * a.dn_sz + head * a.dn_sh;
    const int ncols = min(64, a.X - n0);            // valid columns of this tile (a multiple of 8)

    floatx4 acc[2][4];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = Frag<float>::zero();
    uint16_t* my = vt[w];
    const int p1 = a.seg_ptr[seg + 1];
    for (int p = a.seg_ptr[seg] + w; p < p1; p += 4) {
        const T* blkp = spz + (long)a.seg_blk[p] * 1024;
        const long krow0 = (long)a.seg_inner[p] * 32;
        // dense tile rows krow0..+31, columns n0..n0+63 -> LDS (lane: row 8*it + lane/8, 8 columns)
        uint4 stage[4];
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int k = 8 * it + (lane >> 3), c8 = 8 * (lane & 7);
            stage[it] = make_uint4(0, 0, 0, 0);
            if (c8 < ncols) stage[it] = *reinterpret_cast<const uint4*>(dnp + (krow0 + k) * a.dn_s0 + n0 + c8);
        }
        uint4 fs[2];
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) fs[tm] = *reinterpret_cast<const uint4*>(blkp + (16 * tm + r16) * 32 + 8 * g);
        __builtin_amdgcn_wave_barrier();            // previous iteration's LDS reads are done (in-order DS)
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int k = 8 * it + (lane >> 3), c8 = 8 * (lane & 7);
            uint2* dst = reinterpret_cast<uint2*>(my + k * DSD_LD + c8);
            dst[0] = make_uint2(stage[it].x, stage[it].y);
            dst[1] = make_uint2(stage[it].z, stage[it].w);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) {
            // column n = 16tn + r16 of the tile, rows k = 8g..8g+7
            const uint16_t* src = my + (8 * g) * DSD_LD + 16 * tn + r16;
            uint4 fd;
            fd.x = (uint32_t)src[0] | ((uint32_t)src[DSD_LD] << 16);
            fd.y = (uint32_t)src[2 * DSD_LD] | ((uint32_t)src[3 * DSD_LD] << 16);
            fd.z = (uint32_t)src[4 * DSD_LD] | ((uint32_t)src[5 * DSD_LD] << 16);
            fd.w = (uint32_t)src[6 * DSD_LD] | ((uint32_t)src[7 * DSD_LD] << 16);
            acc[0][tn] = Frag32<T>::mma(fd, fs[0], acc[0][tn]);
            acc[1][tn] = Frag32<T>::mma(fd, fs[1], acc[1][tn]);
        }
    }
    // lane holds C[m = 16tm + r16][n = 16tn + 4g + i]; sum the four waves
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 4; ++tn)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[w][16 * tm + r16][16 * tn + 4 * g + i] = acc[tm][tn][i];
    __syncthreads();
    const int m = tid >> 3, c8 = 8 * (tid & 7);
    if (c8 < ncols) {
        floatx4 lo, hi;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo[i] = (part[0][m][c8 + i] + part[1][m][c8 + i]) + (part[2][m][c8 + i] + part[3][m][c8 + i]);
            hi[i] = (part[0][m][c8 + 4 + i] + part[1][m][c8 + 4 + i]) + (part[2][m][c8 + 4 + i] + part[3][m][c8 + 4 + i]);
        }
        T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh + ((long)brow * 32 + m) * a.c_sm + n0 + c8;
        store4_f32(cp, lo);
        store4_f32(cp + 4, hi);
    }
}

// DSD for layouts whose neighbouring block-rows share most of their columns: one workgroup per
// (batch, head, four consecutive block-rows, 64-column tile of the dense operand), wave w owning
// output rows of block-row 4*group + w -- no split of the reduction, so no partial sums to merge.
// The workgroup walks the union of the four column lists; each 32 x 64 tile of the dense operand
// is loaded once (16-byte global loads) and written to LDS transposed, [column][k], which turns the
// MFMA fragment of a [k][n] operand into one 16-byte LDS read.  Sparse blocks come straight from
// global memory, each read by exactly one wave.  Tiles and sparse fragments of step s+1 are in
// flight while step s is multiplied.
struct DsdUniArgs {
    const void* sp; const void* dn; void* c;
    const int32_t* uni_ptr; const int32_t* uni_inner; const int32_t* uni_blk;
    int per_head, grps_per_head, n_heads, Z, N;
    long sp_sz, dn_sz, dn_sh, dn_sk, c_sz, c_sh, c_sm;
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
};
constexpr int DSDU_LD = 40;     // LDS row stride in elements ([column][k], 32 k + 8): 16 columns hit all banks once

template <typename T, bool TA>     // TA: every sparse block is used transposed (segments are block-columns of the layout)
__global__ __launch_bounds__(256) void bs_dsd32u_kernel(const DsdUniArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t vt[2][64 * DSDU_LD];
    // TA: a wave turns its 32x32 block through a private LDS tile, [column][row]
    __shared__ __attribute__((aligned(16))) uint16_t bt[TA ? 4 : 1][TA ? 32 * DSDU_LD : 8];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ntn = (a.N + 63) / 64;
    int unit, pos;
    if (!unit_of(blockIdx.x, a.n_xcd, a.grps_per_head * ntn, a.n_heads * a.Z, unit, pos)) return;
    const int z = unit / a.n_heads, head = unit % a.n_heads, grp = pos / ntn, n0 = (pos % ntn) * 64;
    const int ug = head * a.grps_per_head + grp;
    const int p0 = a.uni_ptr[ug], n = a.uni_ptr[ug + 1] - p0;
    const int bi = grp * 4 + w;
    const bool have_row = bi < a.per_head;
    const int ncols = min(64, a.N - n0);            // valid columns of this tile (a multiple of 8)
    const T* spz = reinterpret_cast<const T*>(a.sp) + z * a.sp_sz;
    const T* dnp = reinterpret_cast<const T*>(a.dn) + z * a.dn_sz + head * a.dn_sh + n0;

    floatx4 acc[2][4];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = Frag<float>::zero();

    // staging: thread holds dense row k = tid / 8, columns c8 .. c8 + 7.  Column n lands in LDS row
    // 32*(n>>5) + 16*((n>>2)&1) + 4*((n>>3)&3) + (n&3): MFMA tile tn reads LDS rows 16 tn .. 16 tn + 15
    // and its row i is column 32*(tn/2) + 8*(i/4) + 4*(tn%2) + i%4, so tiles 2q and 2q+1 give a lane
    // eight consecutive output columns.
    const int sk = tid >> 3, c8 = 8 * (tid & 7);
    uint4 stage, fs[2], fs_next[2] = {make_uint4(0, 0, 0, 0), make_uint4(0, 0, 0, 0)};
    int blk_next = -1;
    auto fetch = [&](int inner, int blk_id) {
        const long krow0 = (long)inner * 32;
        stage = make_uint4(0, 0, 0, 0);
        if (c8 < ncols) stage = *reinterpret_cast<const uint4*>(dnp + (krow0 + sk) * a.dn_sk + c8);
        blk_next = have_row ? blk_id : -1;
        if (blk_next >= 0) {
            const T* blkp = spz + (long)blk_next * 1024;
#pragma unroll
            for (int tm = 0; tm < 2; ++tm) {
                // every sparse block is read by exactly one wave: nontemporal
                const uintx4 t_ = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(blkp + (16 * tm + r16) * 32 + 8 * g));
                fs_next[tm] = make_uint4(t_[0], t_[1], t_[2], t_[3]);
            }
        }
    };
    auto stash = [&](int buf) {
        const uint32_t v[4] = {stage.x, stage.y, stage.z, stage.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int nn = c8 + i;
            const int lrow = 32 * (nn >> 5) + 16 * ((nn >> 2) & 1) + 4 * ((nn >> 3) & 3) + (nn & 3);
            vt[buf][lrow * DSDU_LD + sk] = (uint16_t)(v[i >> 1] >> (16 * (i & 1)));
        }
    };
    // the index lists are read one step ahead of the fetch that uses them
    int inner_n1 = n > 1 ? a.uni_inner[p0 + 1] : 0, id_n1 = n > 1 ? a.uni_blk[(long)(p0 + 1) * 4 + w] : -1;
    if (n > 0) {
        fetch(a.uni_inner[p0], a.uni_blk[(long)p0 * 4 + w]);
        stash(0);
    }
    drain_loads();
    __syncthreads();
    for (int s = 0; s < n; ++s) {
        const int blk = blk_next;
        fs[0] = fs_next[0];
        fs[1] = fs_next[1];
        const int inner_n2 = s + 2 < n ? a.uni_inner[p0 + s + 2] : 0;
        const int id_n2 = s + 2 < n ? a.uni_blk[(long)(p0 + s + 2) * 4 + w] : -1;
        if (s + 1 < n) fetch(inner_n1, id_n1);
        inner_n1 = inner_n2;
        id_n1 = id_n2;
        if (blk >= 0) {
            if (TA) {
                // the lane holds rows 16 tm + r16 of the block, columns 8g .. 8g + 7: they go to LDS as
                // [column][row] and come back as fragments of the transposed block (a wave-private tile;
                // LDS operations of a wave complete in order)
                uint16_t* my = bt[w];
#pragma unroll
                for (int tm = 0; tm < 2; ++tm) {
                    const uint32_t v[4] = {fs[tm].x, fs[tm].y, fs[tm].z, fs[tm].w};
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        my[(8 * g + e) * DSDU_LD + 16 * tm + r16] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int tm = 0; tm < 2; ++tm) fs[tm] = *reinterpret_cast<const uint4*>(my + (16 * tm + r16) * DSDU_LD + 8 * g);
                __builtin_amdgcn_wave_barrier();
            }
            const uint16_t* tp = vt[s & 1];
#pragma unroll
            for (int tn = 0; tn < 4; ++tn) {
                const uint4 fd = *reinterpret_cast<const uint4*>(tp + (16 * tn + r16) * DSDU_LD + 8 * g);
                acc[0][tn] = Frag32<T>::mma(fd, fs[0], acc[0][tn]);
                acc[1][tn] = Frag32<T>::mma(fd, fs[1], acc[1][tn]);
            }
        }
        if (s + 1 < n) stash((s + 1) & 1);
        __syncthreads();
    }
    if (!have_row) return;
    // lane holds C[m = 16tm + r16][n = 32q + 8g + 4(tn%2) + i], tn = 2q, 2q+1
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh + n0;
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int nn = 32 * q + 8 * g;
            if (nn < ncols) store8_f32(cp + ((long)bi * 32 + 16 * tm + r16) * a.c_sm + nn, acc[tm][2 * q], acc[tm][2 * q + 1]);
        }
}

// ---------------------------------------------------------------------------------------
// DDS: dense = dense x sparse
// ---------------------------------------------------------------------------------------
template <typename T, int BLK>
__global__ __launch_bounds__(256) void bs_dds_kernel(DxdArgs a) {
    constexpr int TILE = BLK >= 32 ? 32 : 16, NTL = TILE / 16, SUBN = BLK / TILE;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const long wid = (long)blockIdx.x * 4 + w;
    const long per_mt = (long)a.n_seg * SUBN;
    const long mt = wid / per_mt;
    if (mt * 32 >= a.X) return;
    const int rem = (int)(wid % per_mt), seg = rem / SUBN, subn = rem % SUBN;
    const int z = blockIdx.y;
    const int head = seg / a.per_head, bcol = seg % a.per_head;
    const long m0 = mt * 32;
    const T* spz = reinterpret_cast<const T*>(a.sp) + z * a.sp_sz;
    const T* dnp = reinterpret_cast<const T*>(a.dn) + z * a.dn_sz + head * a.dn_sh;

    floatx4 acc[2][NTL];
#pragma unroll
    for (int tn = 0; tn < NTL; ++tn) { acc[0][tn] = Frag<float>::zero(); acc[1][tn] = Frag<float>::zero(); }
    bool mok[2];
    mok[0] = m0 + r16 < a.X;
    mok[1] = m0 + 16 + r16 < a.X;

    const int p1 = a.seg_ptr[seg + 1];
    for (int p = a.seg_ptr[seg]; p < p1; ++p) {
        const T* blkp = spz + (long)a.seg_blk[p] * (BLK * BLK);
        const long kcol0 = (long)a.seg_inner[p] * BLK;
#pragma unroll
        for (int kk = 0; kk < BLK; kk += 16) {
            typename Frag<T>::type fs[NTL], fd[2];
#pragma unroll
            for (int tn = 0; tn < NTL; ++tn) {
                const int n = subn * TILE + 16 * tn + r16;
                fs[tn] = a.trans ? Frag<T>::load(blkp + n * BLK + kk + 4 * g)
                                 : Frag<T>::gather(blkp + (kk + 4 * g) * BLK + n, BLK);
            }
#pragma unroll
            for (int tm = 0; tm < 2; ++tm) {
                fd[tm] = Frag<T>::zero();
                if (mok[tm])
                    fd[tm] = frag_at<T>(dnp + (m0 + 16 * tm + r16) * a.dn_s0 + (kcol0 + kk + 4 * g) * a.dn_s1, a.dn_s1);
            }
#pragma unroll
            for (int tn = 0; tn < NTL; ++tn) {
                acc[0][tn] = Frag<T>::mma(fs[tn], fd[0], acc[0][tn]);
                acc[1][tn] = Frag<T>::mma(fs[tn], fd[1], acc[1][tn]);
            }
        }
    }
    // lane holds C[m = m0 + 16tm + r16][n = 16tn + 4g + i]
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh;
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {
        if (!mok[tm]) continue;
        const long m = m0 + 16 * tm + r16;
#pragma unroll
        for (int tn = 0; tn < NTL; ++tn) {
            const long n = (long)bcol * BLK + subn * TILE + 16 * tn + 4 * g;
            if (a.bias) {
                const T* bp = reinterpret_cast<const T*>(a.bias) + (long)head * a.per_head * BLK + n;
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[tm][tn][i] += Elem<T>::to_f32(bp[i]);
            }
            store_tile_row<T>(cp + m * a.c_sm + n * a.c_sn, a.c_sn, acc[tm][tn], 4);
        }
    }
}

// Fast DDS (y = x W^T, W block-sparse, blocks read transposed) for 32x32 blocks of a 2-byte type,
// the Pixelfly linear.  Consecutive output block-rows that reduce over the same input blocks are
// grouped (at most four per group, table built on the host): a group is a small dense GEMM
// y[M x 32g] = x[:, listed input blocks] . W_group^T.  A workgroup owns one group and walks a stream
// of 128-token tiles with one continuous pipeline: per input block the 128 x 32 activation tile and
// the group's 32g x 32 weight tile are staged in LDS (registers hold the next-but-one step's tiles
// while the MFMAs of the current one run, across tile boundaries), the 2 x 2 waves own 64 x 64
// outputs each, form them with 16x16x32 MFMAs and store them after the tile's last input block.
struct DdsGroupArgs {
    const void* sp; const void* dn; void* c;
    const int32_t* seg_ptr; const int32_t* seg_blk; const int32_t* seg_inner;
    const int32_t* grp_row0; const int32_t* grp_n;
    int per_head, M;
    long sp_sz, dn_sz, dn_sh, dn_sm, c_sz, c_sh, c_sm;
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
    int n_grp;          // groups (the weight-stationary kernel deals (token stream, group) pairs itself)
    const void* bias;   // optional: one value per output column, added before the result is rounded
};
constexpr int DDS_MAX_STEPS = 128;   // longest reduction list the tiled kernel accepts
#ifndef FLY_DDS_STATIONARY
#define FLY_DDS_STATIONARY 2         // weight-stationary kernels where the group's weights fit the LDS: 1 = activation
#endif                               // fragments straight from memory, 2 = staged through LDS when there are enough tokens
#ifndef FLY_DDS_DEPTH
#define FLY_DDS_DEPTH 2              // steps (of two input blocks) its activation loads run ahead
#endif
#ifndef FLY_DDS_DIST
#define FLY_DDS_DIST 2               // steps the loads of the 128-token kernel run ahead of its MFMAs
#endif

// eight consecutive values of an optional bias vector, added to b0 | b1
template <typename T>
__device__ __forceinline__ void bias8(const void* bias, long at, floatx4& b0, floatx4& b1) {
    if (bias == nullptr) return;                            // (uniform)
    const T* p = reinterpret_cast<const T*>(bias) + at;
#pragma unroll
    for (int i = 0; i < 4; ++i) { b0[i] += Elem<T>::to_f32(p[i]); b1[i] += Elem<T>::to_f32(p[4 + i]); }
}

template <typename T, bool WT, int DIST = FLY_DDS_DIST>     // WT: blocks are [k][n] (y = x W) and are transposed on their way into LDS
__global__ __launch_bounds__(256) void bs_dds32_kernel(DdsGroupArgs a) {
    // A pipeline step takes TWO entries of the reduction list.  The LDS tiles are [row][64 k] with 128-byte rows, the
    // first entry's 32 inputs in front; the eight 16-byte chunks of a row are stored at chunk ^ ((row >> 1) & 7).  Then
    // both the 16-byte fragment reads (16 consecutive rows, one chunk) and the staging writes (2 rows x 8 chunks per 16
    // lanes) cover all 64 banks.  Neighbouring entries of a list are mostly neighbouring input blocks: a staging wave
    // then reads whole 128-byte lines of eight token rows (a compute unit's vector memory path takes one line about
    // every four cycles whether half of it is used or all of it).
    constexpr int LD = 64;
    extern __shared__ __attribute__((aligned(16))) uint16_t dds_smem[];
    uint16_t (*xs)[128 * LD] = reinterpret_cast<uint16_t (*)[128 * LD]>(dds_smem);
    uint16_t (*ws)[128 * LD] = reinterpret_cast<uint16_t (*)[128 * LD]>(dds_smem + 2 * 128 * LD);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, g = lane >> 4;
    const int wm = w >> 1, wn = w & 1;                      // this wave: tokens 64wm.., outputs 64wn..
    const int z = blockIdx.z;
    // Workgroups go to the XCDs (each with its own L2) round-robin in launch order.  The launch
    // index is re-mapped so that the groups working on one stream of token tiles -- they read the same
    // activations -- run on one XCD, one after the other: stream = n_xcd * (slot / groups) + XCD.
    const int lin = blockIdx.x + gridDim.x * blockIdx.y, slot = lin / a.n_xcd;
    const int grp = slot % (int)gridDim.x, ty = a.n_xcd * (slot / (int)gridDim.x) + lin % a.n_xcd, gy = gridDim.y;   // gridDim.y is a multiple of n_xcd
    // token tiles ty, ty + gy, ... : the group's tables are read once and the load -> LDS -> MFMA
    // pipeline runs on across tile boundaries
    const int tiles_all = (a.M + 127) / 128;
    if (ty >= tiles_all) return;                            // workgroup-uniform
    const int my_tiles = (tiles_all - ty + gy - 1) / gy;
    const int row0 = a.grp_row0[grp], gn = a.grp_n[grp];    // first output block-row (segment) and count
    const int head = row0 / a.per_head, bcol0 = row0 % a.per_head;
    const int p0 = a.seg_ptr[row0], nin = a.seg_ptr[row0 + 1] - p0;
    const uint16_t* spz = reinterpret_cast<const uint16_t*>(a.sp) + z * a.sp_sz;
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.dn) + z * a.dn_sz + head * a.dn_sh;

    // the group's reduction list (inner block per entry, block id per entry and output block-row) is
    // read once into LDS: the per-step loads then depend on no other global load
    __shared__ int s_inner[DDS_MAX_STEPS];
    __shared__ int s_blk[4][DDS_MAX_STEPS];
    for (int i = tid; i < nin; i += 256) s_inner[i] = a.seg_inner[p0 + i];
    for (int i = tid; i < 4 * nin; i += 256) {
        const int ob = i / nin, t = i % nin;
        s_blk[ob][t] = ob < gn ? a.seg_blk[a.seg_ptr[row0 + ob] + t] : -1;
    }
    __syncthreads();

    // staging roles: thread -> (row = tid/8 + 32 hh, 16-byte chunk = tid%8) of the x and W tiles; chunks 0..3 belong
    // to the step's first entry, 4..7 to its second
    const int srow = tid >> 3, sc = tid & 7, sel = sc >> 2, schunk = (sc & 3) * 8;
    const int npair = (nin + 1) / 2;
    const int n_steps = my_tiles * npair;
    // DIST register sets: the loads of step s+DIST are issued while step s computes and are parked in LDS
    // one iteration before they are used
    // (native vectors: arrays of the uint4 struct passed by reference do not stay in registers)
    // Every fetch issues the same number of loads on every path (a step past the end re-reads the last
    // one, an absent weight block reads block 0 and is zeroed when it is parked): only then can the
    // compiler count how many newer loads may stay in flight when it waits for the older set.
    uintx4 rx[DIST][4], rw[DIST][4];                        // set j holds the steps congruent to j modulo DIST
    bool wl[DIST][4];                                       // weight block present?
    int f_tile = 0, f_t = 0;                                // fetch cursor: (token tile, step inside it)
    // A load is "base + per-thread byte offset": the two input blocks of a step and the weight blocks of its eight
    // (output block, entry) pairs come out of LDS once through the first lane; a thread picks the entry its chunk
    // belongs to; the per-thread offsets change only with the token tile.
    const uint32_t woff = (uint32_t)((srow * 32 + schunk) * 2);
    uint32_t xoff[4] = {0, 0, 0, 0};
    auto fetch = [&](uintx4 (&rx)[4], uintx4 (&rw)[4], bool (&wl)[4]) __attribute__((always_inline)) {
        const bool live = f_tile < my_tiles;                 // past the end: re-read the last step, zero weights
        const int tc = live ? f_t : npair - 1;
        if (f_t == 0) {
            const long m0 = ((long)ty + (long)min(f_tile, my_tiles - 1) * gy) * 128;
#pragma unroll
            for (int hh = 0; hh < 4; ++hh) {
                const long m = min(m0 + srow + 32 * hh, (long)a.M - 1);          // clamped: masked at the store
                xoff[hh] = (uint32_t)((m * a.dn_sm + schunk) * 2);
            }
        }
        const int t0 = 2 * tc, t1 = min(2 * tc + 1, nin - 1);
        const bool second = 2 * tc + 1 < nin;                // an odd list's last step: its second entry is absent
        const int in0 = __builtin_amdgcn_readfirstlane(s_inner[t0]), in1 = __builtin_amdgcn_readfirstlane(s_inner[t1]);
        const char* xb = reinterpret_cast<const char*>(xp + (long)(sel ? in1 : in0) * 32);
#pragma unroll
        for (int hh = 0; hh < 4; ++hh) {
            rx[hh] = *reinterpret_cast<const uintx4*>(xb + xoff[hh]);
            const int b0 = __builtin_amdgcn_readfirstlane(s_blk[hh][t0]), b1 = __builtin_amdgcn_readfirstlane(s_blk[hh][t1]);
            const int blk_id = sel ? (second ? b1 : -1) : b0;
            wl[hh] = live && blk_id >= 0;                    // a missing block contributes zero weights
            rw[hh] = *reinterpret_cast<const uintx4*>(reinterpret_cast<const char*>(spz + (long)max(blk_id, 0) * 1024) + woff);
        }
        if (++f_t == npair) { f_t = 0; ++f_tile; }
    };
    // The weight tile sits in LDS in the order the MFMAs read it: row 64*(n/64) + 16*i + r holds output
    // n = 64*(n/64) + 32*(i/2) + 8*(r/4) + 4*(i%2) + r%4, so that a wave's fragment read walks 16
    // consecutive LDS rows.
    auto wrow = [](int n) { const int b = n & 31; return (n & 64) + 16 * (2 * ((n >> 5) & 1) + ((b >> 2) & 1)) + 4 * (b >> 3) + (b & 3); };
    auto slot_of = [](int row, int chunk) { return row * LD + 8 * (chunk ^ ((row >> 1) & 7)); };
    auto stash = [&](int buf, const uintx4 (&rx)[4], const uintx4 (&rw)[4], const bool (&wl)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int hh = 0; hh < 4; ++hh) {
            *reinterpret_cast<uintx4*>(&xs[buf][slot_of(srow + 32 * hh, sc)]) = rx[hh];
            const uintx4 wv = wl[hh] ? rw[hh] : uintx4{0, 0, 0, 0};
            if (!WT) {
                // block row srow of output block hh, inputs schunk .. of entry `sel`
                *reinterpret_cast<uintx4*>(&ws[buf][slot_of(wrow(32 * hh + srow), sc)]) = wv;
            } else {
                // the thread holds row k = srow of the block [k][n], columns n = schunk .. schunk + 7: the
                // LDS tile is [n][k] either way, so these eight go out one by one
                const int kk = 32 * sel + srow;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int n = wrow(32 * hh + schunk + e);
                    ws[buf][slot_of(n, kk >> 3) + (kk & 7)] = (uint16_t)(wv[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
    };

    floatx4 acc[4][4];
#pragma unroll
    for (int tm = 0; tm < 4; ++tm)
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = Frag<float>::zero();
    const bool wave_active = 2 * wn < gn;                   // its output blocks exist in this group

    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh;
    // lane holds y[m = 64wm + 16tm + r16][n = 32*(output block) + 8g + 4*(tn%2) + i]: 16-byte stores
    auto store_tile = [&](int tile) __attribute__((always_inline)) {
        const long m0 = ((long)ty + (long)tile * gy) * 128;
#pragma unroll
        for (int tm = 0; tm < 4; ++tm) {
            const long m = m0 + 64 * wm + 16 * tm + r16;
#pragma unroll
            for (int o2 = 0; o2 < 2; ++o2) {
                const int ob = 2 * wn + o2;
                if (m < a.M && ob < gn) {
                    const long n = (long)(bcol0 + ob) * 32 + 8 * g;
                    floatx4 b0 = Frag<float>::zero(), b1 = Frag<float>::zero();
                    bias8<T>(a.bias, head * (long)a.per_head * 32 + n, b0, b1);
                    store8_f32(cp + m * a.c_sm + n, acc[tm][2 * o2] + b0, acc[tm][2 * o2 + 1] + b1);
                }
            }
#pragma unroll
            for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = Frag<float>::zero();
        }
    };
    int c_tile = 0, c_t = 0;                                // compute cursor
    // this lane's 16 bytes inside a 16-row fragment, per entry of the step (fragments start at multiples of 16 rows)
    const int frag_off[2] = {r16 * LD + 8 * (g ^ (r16 >> 1)), r16 * LD + 8 * ((4 + g) ^ (r16 >> 1))};
    auto compute = [&](int cur) __attribute__((always_inline)) {
        if (wave_active) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                uint4 fx[4], fw[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    fx[i] = *reinterpret_cast<const uint4*>(&xs[cur][(64 * wm + 16 * i) * LD + frag_off[kb]]);
                    // W-tile i covers output block i/2; its MFMA row r is block row 8*(r/4) + 4*(i%2) + r%4
                    fw[i] = *reinterpret_cast<const uint4*>(&ws[cur][(64 * wn + 16 * i) * LD + frag_off[kb]]);
                }
#pragma unroll
                for (int tm = 0; tm < 4; ++tm)
#pragma unroll
                    for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = Frag32<T>::mma(fw[tn], fx[tm], acc[tm][tn]);
            }
            if (++c_t == npair) { store_tile(c_tile); c_t = 0; ++c_tile; }   // the tile's last entries
        }
    };
    if (nin == 0) {                                         // no input block: zero rows
        if (wave_active)
            for (int tile = 0; tile < my_tiles; ++tile) store_tile(tile);
        return;
    }
    // Loads run DIST steps ahead of the MFMAs in DIST register sets: a step's tiles are asked for, parked in LDS
    // DIST - 1 iterations later (one iteration before they are used), and every global load has that long to arrive.
    // The loop is unrolled over the least common multiple of the two LDS stages and the DIST sets, so that every
    // register set and stage index is a constant.
#pragma unroll
    for (int j = 0; j < DIST; ++j) fetch(rx[j], rw[j], wl[j]);
    drain_loads_but<8 * (DIST - 1)>();                       // set 0 has arrived
    stash(0, rx[0], rw[0], wl[0]);
    __syncthreads();
    constexpr int U = (DIST % 2 == 0) ? DIST : 2 * DIST;
    for (int step = 0; step < n_steps; step += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // (no early exit inside: every path through the body issues the same loads, so the compiler can count how
            //  many newer ones may stay in flight when it waits for a set)
            fetch(rx[u % DIST], rw[u % DIST], wl[u % DIST]);                    // step + u + DIST; its set was parked an iteration ago
            if (step + u < n_steps) compute(u & 1);
            stash((u + 1) & 1, rx[(u + 1) % DIST], rw[(u + 1) % DIST], wl[(u + 1) % DIST]);
            drain_loads_but<8 * (DIST - 1)>();              // the set parked next iteration has arrived
            __syncthreads();
        }
    }
}

// DDS for few tokens, 32 x 32 blocks of a 2-byte type.  The grouped kernel above gives a workgroup 128 tokens and up to
// four block-rows: one image of 196 tokens through the narrowing layer of a channel MLP (24 block-rows of 36 blocks) left 16
// workgroups that walk the whole list, 20.2 us; 7.6 us here.  Here a workgroup owns 32 tokens of ONE block-row and its eight waves share the reduction list
// (wave w: entries w, w + 8, ...), operands straight from memory in MFMA order, the loads of four entries in flight; the
// partial sums meet in LDS.  What bounds it is the latency of two dependent loads and the reduction.
template <typename T, bool WT>
__global__ __launch_bounds__(512) void bs_dds32w_kernel(DdsGroupArgs a) {
    constexpr int NW = 8, AHEAD = 4;
    __shared__ __attribute__((aligned(16))) floatx4 red[NW][4][64];             // [wave][token half, output half][lane]
    __shared__ __attribute__((aligned(16))) uint16_t wt[WT ? NW : 1][WT ? AHEAD : 1][WT ? 32 * 32 : 8];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int seg = blockIdx.x, z = blockIdx.z, head = seg / a.per_head, bcol = seg % a.per_head;
    const long m0 = (long)blockIdx.y * 32;
    const int p0 = a.seg_ptr[seg], nin = a.seg_ptr[seg + 1] - p0;
    const uint16_t* spz = reinterpret_cast<const uint16_t*>(a.sp) + z * a.sp_sz;
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.dn) + z * a.dn_sz + head * a.dn_sh;
    const uint16_t* xrow[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) xrow[i] = xp + min(m0 + 16 * i + r16, (long)a.M - 1) * a.dn_sm;         // clamped: masked at the store
    // products are formed transposed, weight rows dealt so that result row 4 g + i of half j is output 8 g + 4 j + i: a
    // lane ends up with eight consecutive outputs of one token
    floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) { acc[i][0] = Frag<float>::zero(); acc[i][1] = Frag<float>::zero(); }
    const int mine = (nin - w + NW - 1) / NW;                                  // (w < NW: >= 0)
    for (int t0 = 0; t0 < mine; t0 += 64) {
        const int at = p0 + min(w + NW * (t0 + lane), nin - 1);                // this wave's next 64 entries, one a lane
        const int l_in = a.seg_inner[at], l_blk = a.seg_blk[at];
        const int nt = min(mine - t0, 64);
        for (int t = 0; t < nt; t += AHEAD) {
            uintx4 fx[AHEAD][2], fw[AHEAD][2];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {                                  // (past the end: the last entry again, not used)
                const int tu = min(t + u, nt - 1);
                const long in0 = (long)__builtin_amdgcn_readlane(l_in, tu) * 32;
                const uint16_t* blk = spz + (long)__builtin_amdgcn_readlane(l_blk, tu) * 1024;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (!WT) {
                        fx[u][i] = *reinterpret_cast<const uintx4*>(xrow[i] + in0 + 8 * g);
                        fw[u][i] = *reinterpret_cast<const uintx4*>(blk + (8 * (r16 >> 2) + 4 * i + (r16 & 3)) * 32 + 8 * g);
                    } else {                                                   // contraction slots {4 g + i, 16 + 4 g + i}
                        const uint2 lo = *reinterpret_cast<const uint2*>(xrow[i] + in0 + 4 * g), hi = *reinterpret_cast<const uint2*>(xrow[i] + in0 + 16 + 4 * g);
                        fx[u][i] = uintx4{lo.x, lo.y, hi.x, hi.y};
                        fw[u][i] = *reinterpret_cast<const uintx4*>(blk + 8 * lane + 512 * i);
                    }
                }
            }
            if (WT) {                                                          // [k][n] blocks: transposed by LDS reads of the wave's own copy
#pragma unroll
                for (int u = 0; u < AHEAD; ++u)
#pragma unroll
                    for (int i = 0; i < 2; ++i) *reinterpret_cast<uintx4*>(&wt[WT ? w : 0][WT ? u : 0][WT ? 8 * lane + 512 * i : 0]) = fw[u][i];
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // (read back by other lanes of the wave only)
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int u = 0; u < AHEAD; ++u)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const uint16_t* q = &wt[WT ? w : 0][WT ? u : 0][WT ? (4 * g + (r16 >> 2)) * 32 + 8 * (r16 & 3) + 4 * j : 0];
                        fw[u][j] = lds_read_tr8(reinterpret_cast<const char*>(q), reinterpret_cast<const char*>(q + (WT ? 16 * 32 : 0)));
                    }
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (t + u < nt) {                                              // (wave-uniform)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j) acc[i][j] = mma32<T>(fw[u][j], fx[u][i], acc[i][j]);
                }
            if (WT) { asm volatile("" ::: "memory"); __builtin_amdgcn_wave_barrier(); }
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) red[w][2 * i + j][lane] = acc[i][j];
    __syncthreads();
    if (w < 2) {                                                               // wave i finishes token half i
        floatx4 s0 = Frag<float>::zero(), s1 = Frag<float>::zero();
        bias8<T>(a.bias, (long)seg * 32 + 8 * g, s0, s1);
#pragma unroll
        for (int v = 0; v < NW; ++v) { s0 += red[v][2 * w][lane]; s1 += red[v][2 * w + 1][lane]; }
        const long m = m0 + 16 * w + r16;
        if (m < a.M) store8_f32(reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh + m * a.c_sm + (long)bcol * 32 + 8 * g, s0, s1);
    }
}

// Weight-stationary DDS for groups whose weights fit the LDS (reduction lists of up to 9 input blocks: layers that
// widen, such as the first linear of a channel MLP).  The group's weight tiles -- the same for every token tile -- are
// brought into LDS once; after that a wave needs nothing from its neighbours: it owns 64 tokens against all outputs of
// the group, takes its activation fragments STRAIGHT from global memory in MFMA operand order (lane (r, g): token r,
// inputs 8 g .. 8 g + 7 of the step's block, 16 contiguous bytes), DEPTH steps ahead in DEPTH register sets, and reads
// the step's weight fragments from LDS.  No barrier in the loop, no activation staging, no weight traffic per token
// tile; every weight fragment read feeds four MFMAs.  Tokens are the rows of the products and the weight tiles are
// dealt so that tile n holds outputs 8 r + n (r = 0..15): a lane then ends up with eight CONSECUTIVE outputs of four
// tokens, and one store instruction writes four whole 256-byte rows of the result (with 64-byte pieces per row the
// stores of the 308 MB result were 40 % of the kernel's time).  Two workgroups of four waves per compute unit; the
// (token stream, group) pairs are dealt to the XCDs in contiguous runs, so that the groups reading one stream's
// activations share an L2.
constexpr int DDS_STAT_STEPS = 9;         // longest reduction list: 8 KB of weight tiles per step, 72 KB, two workgroups per CU

template <typename T, bool WT, int DEPTH>
__global__ __launch_bounds__(256) void bs_dds32s_kernel(DdsGroupArgs a, int n_streams) {
    constexpr int STEP = 8 * 16 * 32;                       // elements of a step's eight weight tiles
    extern __shared__ __attribute__((aligned(16))) uint16_t wres[];     // [step][tile n][row r][32 k]: output 8 r + n of the group
    __shared__ int s_inner[DDS_STAT_STEPS];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, g = lane >> 4;
    const int z = blockIdx.y;
    // pair index: the dispatcher deals workgroup ids to the XCDs in turn; XCD x takes the pairs x * per_xcd ...
    const int per_xcd = (int)gridDim.x / a.n_xcd;
    const int pair = ((int)blockIdx.x % a.n_xcd) * per_xcd + (int)blockIdx.x / a.n_xcd;
    const int n_grp = a.n_grp;
    if (pair >= n_streams * n_grp) return;                  // workgroup-uniform
    const int ty = pair / n_grp, grp = pair % n_grp, gy = n_streams;
    const int tiles_all = (a.M + 255) / 256;
    if (ty >= tiles_all) return;
    const int my_tiles = (tiles_all - ty + gy - 1) / gy;
    const int row0 = a.grp_row0[grp], gn = a.grp_n[grp];
    const int head = row0 / a.per_head, bcol0 = row0 % a.per_head;
    const int p0 = a.seg_ptr[row0], nin = a.seg_ptr[row0 + 1] - p0;
    const uint16_t* spz = reinterpret_cast<const uint16_t*>(a.sp) + z * a.sp_sz;
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.dn) + z * a.dn_sz + head * a.dn_sh;
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh;

    for (int i = tid; i < nin; i += 256) s_inner[i] = a.seg_inner[p0 + i];
    // the group's weights, once (output blocks the group lacks: zeros)
    for (int idx = tid; idx < nin * 512; idx += 256) {
        const int chunk = idx & 3, row = (idx >> 2) & 31, ob = (idx >> 7) & 3, t = idx >> 9;
        const int blk_id = ob < gn ? a.seg_blk[a.seg_ptr[row0 + ob] + t] : -1;
        uintx4 v = {0, 0, 0, 0};
        if (blk_id >= 0) v = *reinterpret_cast<const uintx4*>(spz + (long)blk_id * 1024 + row * 32 + chunk * 8);
        uint16_t* dst = wres + (size_t)t * STEP;
        if (!WT) {
            // block row `row` is output 32 ob + row: tile row % 8, row 4 ob + row / 8; the thread's 8 inputs stay together
            *reinterpret_cast<uintx4*>(dst + (row & 7) * 512 + (4 * ob + (row >> 3)) * 32 + 8 * chunk) = v;
        } else {
            // the block is [input][output]: the thread holds input `row`, outputs 32 ob + 8 chunk + e -> tile e, row 4 ob + chunk
#pragma unroll
            for (int e = 0; e < 8; ++e)
                dst[e * 512 + (4 * ob + chunk) * 32 + row] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
    }
    __syncthreads();

    const bool col_live = 8 * r16 < 32 * gn;                // this lane's eight outputs exist in the group
    floatx4 bias_lo = Frag<float>::zero(), bias_hi = Frag<float>::zero();       // what the sums start from
    if (col_live) bias8<T>(a.bias, ((long)head * a.per_head + bcol0) * 32 + 8 * r16, bias_lo, bias_hi);
    floatx4 acc[4][8];
    auto reset = [&](int tm) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const float x = n < 4 ? bias_lo[n & 3] : bias_hi[n & 3];
            acc[tm][n] = floatx4{x, x, x, x};
        }
    };
#pragma unroll
    for (int tm = 0; tm < 4; ++tm) reset(tm);
    // lane holds y[m = 64 w + 16 tm + 4 g + i][n0 + 8 r16 .. + 7]: one 16-byte store per (tm, i), 256 bytes per row and
    // instruction
    auto store_tile = [&](int tile) __attribute__((always_inline)) {
        const long m0 = ((long)ty + (long)tile * gy) * 256 + 64 * w + 4 * g;
        T* base = cp + (long)bcol0 * 32 + 8 * r16;
#pragma unroll
        for (int tm = 0; tm < 4; ++tm) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const long m = m0 + 16 * tm + i;
                if (m < a.M && col_live) {
                    const floatx4 lo = {acc[tm][0][i], acc[tm][1][i], acc[tm][2][i], acc[tm][3][i]};
                    const floatx4 hi = {acc[tm][4][i], acc[tm][5][i], acc[tm][6][i], acc[tm][7][i]};
                    store8_f32(base + m * a.c_sm, lo, hi);
                }
            }
            reset(tm);
        }
    };
    if (nin == 0) {                                         // no input block: zero rows
        for (int tile = 0; tile < my_tiles; ++tile) store_tile(tile);
        return;
    }

    // a step takes two entries of the reduction list: neighbouring input blocks share their 128-byte lines, and asked for
    // together the second block's loads find them on their way (a step apart they had left the L1 again)
    const int npair = (nin + 1) / 2;
    const int n_steps = my_tiles * npair;
    uintx4 fx[DEPTH][2][4];
    int f_tile = 0, f_t = 0;                                // fetch cursor: (token tile, pair of entries inside it)
    uint32_t xoff[4] = {0, 0, 0, 0};
    auto fetch = [&](uintx4 (&rx)[2][4]) __attribute__((always_inline)) {
        const int tp = f_tile < my_tiles ? f_t : npair - 1; // past the end: re-read the last step (never used)
        if (f_t == 0) {
            const long m0 = ((long)ty + (long)min(f_tile, my_tiles - 1) * gy) * 256 + 64 * w;
#pragma unroll
            for (int tm = 0; tm < 4; ++tm) {
                const long m = min(m0 + 16 * tm + r16, (long)a.M - 1);           // clamped: masked at the store
                xoff[tm] = (uint32_t)((m * a.dn_sm + 8 * g) * 2);
            }
        }
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {                    // (an odd list's last step reads its last entry twice and uses it once)
            const int inner = __builtin_amdgcn_readfirstlane(s_inner[min(2 * tp + hf, nin - 1)]);
            const char* xb = reinterpret_cast<const char*>(xp + (long)inner * 32);
#pragma unroll
            for (int tm = 0; tm < 4; ++tm) rx[hf][tm] = *reinterpret_cast<const uintx4*>(xb + xoff[tm]);
        }
        if (++f_t == npair) { f_t = 0; ++f_tile; }
    };
    int c_tile = 0, c_t = 0;                                // compute cursor
    const int frag_off = r16 * 32 + 8 * g;                  // this lane's 16 bytes of a weight tile: a wave reads its 1 KB in lane order
    auto compute = [&](const uintx4 (&rx)[2][4]) __attribute__((always_inline)) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            if (2 * c_t + hf < nin) {                       // workgroup-uniform
                const uint16_t* wt = wres + (size_t)(2 * c_t + hf) * STEP + frag_off;
#pragma unroll
                for (int n = 0; n < 8; ++n) {
                    const uint4 fw = *reinterpret_cast<const uint4*>(wt + n * 512);
#pragma unroll
                    for (int tm = 0; tm < 4; ++tm)
                        acc[tm][n] = Frag32<T>::mma(__builtin_bit_cast(uint4, rx[hf][tm]), fw, acc[tm][n]);
                }
            }
        }
        if (++c_t == npair) { store_tile(c_tile); c_t = 0; ++c_tile; }   // the tile's last entries: results out
    };
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) fetch(fx[j]);
    for (int step = 0; step < n_steps; step += DEPTH) {
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            if (step + u < n_steps) compute(fx[u]);
            fetch(fx[u]);                                   // step + u + DEPTH
        }
    }
}

// The weight-stationary DDS with the activations staged through LDS by direct-to-LDS transfers.  A compute unit's
// vector memory path takes about one 128-byte line every four cycles whether half of the line is asked for or all of
// it, and bs_dds32s_kernel's fragment loads (64-byte pieces of 16 token rows per instruction) are what bounds it.  Here
// a wave fetches a step's two input blocks of its 64 tokens as whole 128-byte pieces of token rows (eight rows per
// instruction, the two blocks side by side when they are neighbours) into a stage of its own, 8 KB, and reads the MFMA
// fragments from there.  One workgroup of eight waves per compute unit shares the group's weights (72 KB) and leaves
// room for the eight stages; a wave touches no other wave's stage, so the loop has no barrier: it waits for its
// transfer, reads the step's fragments into registers, starts the next step's transfer into the same stage and then
// multiplies.  16-byte chunk c of token t sits at chunk c ^ ((t >> 1) & 7) of the token's 128 bytes: the transfer
// writes lane by lane, so the lane asks for the chunk that belongs in its slot, and the 16 lanes of a fragment read
// cover all 64 banks.
template <typename T, bool WT>
__global__ __launch_bounds__(512) void bs_dds32d_kernel(DdsGroupArgs a, int n_streams) {
    constexpr int STEP = 8 * 16 * 32;                       // elements of a step's eight weight tiles
    constexpr int WBYTES = DDS_STAT_STEPS * 8192;           // the weights' share of the LDS
    extern __shared__ __attribute__((aligned(1024))) uint16_t wres[];   // [step][tile n][row r][32 k], then 8 stages of 8 KB
    __shared__ int s_inner[DDS_STAT_STEPS];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = blockIdx.y;
    const int per_xcd = (int)gridDim.x / a.n_xcd;
    const int pair = ((int)blockIdx.x % a.n_xcd) * per_xcd + (int)blockIdx.x / a.n_xcd;
    const int n_grp = a.n_grp;
    if (pair >= n_streams * n_grp) return;                  // workgroup-uniform
    const int ty = pair / n_grp, grp = pair % n_grp, gy = n_streams;
    const int tiles_all = (a.M + 511) / 512;
    if (ty >= tiles_all) return;
    const int my_tiles = (tiles_all - ty + gy - 1) / gy;
    const int row0 = a.grp_row0[grp], gn = a.grp_n[grp];
    const int head = row0 / a.per_head, bcol0 = row0 % a.per_head;
    const int p0 = a.seg_ptr[row0], nin = a.seg_ptr[row0 + 1] - p0;
    const uint16_t* spz = reinterpret_cast<const uint16_t*>(a.sp) + z * a.sp_sz;
    const uint16_t* xp = reinterpret_cast<const uint16_t*>(a.dn) + z * a.dn_sz + head * a.dn_sh;
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh;

    for (int i = tid; i < nin; i += 512) s_inner[i] = a.seg_inner[p0 + i];
    for (int idx = tid; idx < nin * 512; idx += 512) {      // the group's weights, once (see bs_dds32s_kernel)
        const int chunk = idx & 3, row = (idx >> 2) & 31, ob = (idx >> 7) & 3, t = idx >> 9;
        const int blk_id = ob < gn ? a.seg_blk[a.seg_ptr[row0 + ob] + t] : -1;
        uintx4 v = {0, 0, 0, 0};
        if (blk_id >= 0) v = *reinterpret_cast<const uintx4*>(spz + (long)blk_id * 1024 + row * 32 + chunk * 8);
        uint16_t* dst = wres + (size_t)t * STEP;
        if (!WT) {
            *reinterpret_cast<uintx4*>(dst + (row & 7) * 512 + (4 * ob + (row >> 3)) * 32 + 8 * chunk) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                dst[e * 512 + (4 * ob + chunk) * 32 + row] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
    }
    __syncthreads();

    const bool col_live = 8 * r16 < 32 * gn;                // this lane's eight outputs exist in the group
    floatx4 bias_lo = Frag<float>::zero(), bias_hi = Frag<float>::zero();       // what the sums start from
    if (col_live) bias8<T>(a.bias, ((long)head * a.per_head + bcol0) * 32 + 8 * r16, bias_lo, bias_hi);
    floatx4 acc[4][8];
    auto reset = [&](int tm) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const float x = n < 4 ? bias_lo[n & 3] : bias_hi[n & 3];
            acc[tm][n] = floatx4{x, x, x, x};
        }
    };
#pragma unroll
    for (int tm = 0; tm < 4; ++tm) reset(tm);
    auto store_tile = [&](int tile) __attribute__((always_inline)) {
        const long m0 = ((long)ty + (long)tile * gy) * 512 + 64 * w + 4 * g;
        T* base = cp + (long)bcol0 * 32 + 8 * r16;
#pragma unroll
        for (int tm = 0; tm < 4; ++tm) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const long m = m0 + 16 * tm + i;
                if (m < a.M && col_live) {
                    const floatx4 lo = {acc[tm][0][i], acc[tm][1][i], acc[tm][2][i], acc[tm][3][i]};
                    const floatx4 hi = {acc[tm][4][i], acc[tm][5][i], acc[tm][6][i], acc[tm][7][i]};
                    store8_f32(base + m * a.c_sm, lo, hi);
                }
            }
            reset(tm);
        }
    };
    if (nin == 0) {                                         // no input block: zero rows
        for (int tile = 0; tile < my_tiles; ++tile) store_tile(tile);
        return;
    }

    const int npair = (nin + 1) / 2;
    const int n_steps = my_tiles * npair;
    char* stage = reinterpret_cast<char*>(wres) + WBYTES + 8192 * w;
    // transfer j of a step brings tokens 8 j .. 8 j + 7 of the wave: this lane's slot is chunk slot lane % 8 of token
    // 8 j + lane / 8, i.e. chunk (lane % 8) ^ ((token >> 1) & 7) of that token's two blocks
    const int tl = lane >> 3;
    uint32_t xoff[8];
    int sel[8];                                             // which of the step's two blocks the lane's chunk belongs to
#pragma unroll
    for (int j = 0; j < 8; ++j) { xoff[j] = 0; sel[j] = 0; }
    int f_tile = 0, f_t = 0;                                // transfer cursor: (token tile, pair of entries inside it)
    auto transfer = [&]() __attribute__((always_inline)) {
        if (f_t == 0) {
            const long m0 = ((long)ty + (long)f_tile * gy) * 512 + 64 * w;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int t = 8 * j + tl, c = (lane & 7) ^ ((t >> 1) & 7);
                const long m = min(m0 + t, (long)a.M - 1);                       // clamped: masked at the store
                xoff[j] = (uint32_t)((m * a.dn_sm + 8 * (c & 3)) * 2);
                sel[j] = c >> 2;
            }
        }
        const int in0 = __builtin_amdgcn_readfirstlane(s_inner[2 * f_t]);
        const int in1 = __builtin_amdgcn_readfirstlane(s_inner[min(2 * f_t + 1, nin - 1)]);   // (an odd list's last step: twice the same)
        const char* xb = reinterpret_cast<const char*>(xp);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            dma_to_lds(xb + xoff[j] + (uint32_t)((sel[j] ? in1 : in0) * 64), stage + 1024 * j);
        if (++f_t == npair) { f_t = 0; ++f_tile; }
    };
    int c_tile = 0, c_t = 0;                                // compute cursor
    const int wfrag = r16 * 32 + 8 * g;                     // this lane's 16 bytes of a weight tile
    // fragment of (token 16 tm + r16, block hf): chunk 4 hf + g, stored at chunk ^ ((token >> 1) & 7)
    int xfrag[2][4];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int tm = 0; tm < 4; ++tm) {
            const int t = 16 * tm + r16;
            xfrag[hf][tm] = t * 128 + 16 * ((4 * hf + g) ^ ((t >> 1) & 7));
        }
    transfer();
    for (int step = 0; step < n_steps; ++step) {
        drain_loads();                                      // this step's activations are in the stage
        uintx4 fx[2][4];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int tm = 0; tm < 4; ++tm) fx[hf][tm] = *reinterpret_cast<const uintx4*>(stage + xfrag[hf][tm]);
        __builtin_amdgcn_s_waitcnt(0xC07F);                 // lgkmcnt(0): the fragments are in registers, the stage is free
        if (step + 1 < n_steps) transfer();                 // (workgroup-uniform) flies under the products below
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            if (2 * c_t + hf < nin) {                       // workgroup-uniform
                const uint16_t* wt = wres + (size_t)(2 * c_t + hf) * STEP + wfrag;
#pragma unroll
                for (int n = 0; n < 8; ++n) {
                    const uint4 fw = *reinterpret_cast<const uint4*>(wt + n * 512);
#pragma unroll
                    for (int tm = 0; tm < 4; ++tm)
                        acc[tm][n] = Frag32<T>::mma(__builtin_bit_cast(uint4, fx[hf][tm]), fw, acc[tm][n]);
                }
            }
        }
        if (++c_t == npair) { store_tile(c_tile); c_t = 0; ++c_tile; }
    }
}

// The same per-wave scheme for reduction lists that do not fit the LDS (layers that narrow: 36 input blocks per output
// block in the second linear of a channel MLP, and the input gradients of layers that widen).  The group's weights pass
// through LDS two list entries (16 KB) at a time, double-buffered and shared by the eight waves, the activations through two
// stages per wave: a step's 8 KB are asked for two steps ahead, its weights one, all straight into LDS.  What bounds it is
// the latency of those transfers between two barriers -- with one stage per wave, weights through registers and [k][n] blocks
// transposed by 16-bit LDS writes a step took 5500 cycles for 1536 of MFMA on its SIMD, now 4400.  (Even shares of the tokens with a
// lower last tile, 256 workgroups for 200 in the case below, made the kernel alone 9 % shorter and the training step no faster.)
// Input gradient of 768 -> 3072 features, 50176 tokens: training step 443 -> 418 us; forward of 3072 -> 768: 492 -> 470 us a step.
// The 160 KB of LDS are full, so the lists are read as scalars.  Weight blocks lie as in memory, 64 bytes a row with 16-byte
// chunk c at c ^ ((row >> 2) & 3), and are the row operand of the products: [n][k] blocks by 16-byte reads, [k][n] blocks by
// transposing reads.  A lane ends up with four consecutive outputs of a token in each tile of 16; a row swap makes eight of two.
constexpr int DDS_PIPE_LDS = 2 * 16384 + 2 * 8 * 8192;

// One group of GN output blocks (a constant: a branch per output block would wait for its weights in turn)
template <typename T, bool WT, int GN>
__device__ __forceinline__ void dds32c_group(const DdsGroupArgs& a, char* lds, int grp, int ty, int gy) {
    constexpr int NT = 2 * GN, TM = 4, NX = 2 * TM;         // NX: a step's transfers of activations per wave
    const int n_tiles = ((a.M + 511) / 512 - ty + gy - 1) / gy;
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = blockIdx.y;
    const int row0 = a.grp_row0[grp];
    const int head = row0 / a.per_head, bcol0 = row0 % a.per_head;
    const int p0 = a.seg_ptr[row0], nin = a.seg_ptr[row0 + 1] - p0;
    const char* spz = reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.sp) + z * a.sp_sz);
    const char* xb = reinterpret_cast<const char*>(reinterpret_cast<const uint16_t*>(a.dn) + z * a.dn_sz + head * a.dn_sh);
    T* cp = reinterpret_cast<T*>(a.c) + z * a.c_sz + head * a.c_sh + (long)bcol0 * 32;

    // outputs 16 n + 4 g .. + 3 of the group, tokens 16 tm + r16
    floatx4 acc[TM][NT];
    // what the sums start from, as it lies in memory (WT: zero, gradients have no bias)
    uint2 bias[WT ? 1 : NT];
#pragma unroll
    for (int n = 0; n < (WT ? 0 : NT); ++n) {
        bias[n] = make_uint2(0u, 0u);
        if (a.bias) {
            const uint16_t* b = reinterpret_cast<const uint16_t*>(a.bias) + ((long)head * a.per_head + bcol0) * 32 + 16 * n + 4 * g;
            bias[n] = make_uint2(b[0] | ((uint32_t)b[1] << 16), b[2] | ((uint32_t)b[3] << 16));
        }
    }
    auto reset = [&](int tm) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if (WT) acc[tm][n] = Frag<float>::zero();
            else {
                const uint2 b = bias[WT ? 0 : n];
                auto one = [](uint32_t bits) __attribute__((always_inline)) { return Elem<T>::to_f32(__builtin_bit_cast(T, (uint16_t)bits)); };
                acc[tm][n] = floatx4{one(b.x & 0xffffu), one(b.x >> 16), one(b.y & 0xffffu), one(b.y >> 16)};
            }
        }
    };
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) reset(tm);
    auto store_tile = [&](int tile) __attribute__((always_inline)) {
        const long m0 = ((long)ty + (long)tile * gy) * 512 + 64 * w + r16;
        T* base = cp + 16 * (g & 1) + 8 * (g >> 1);
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const long m = m0 + 16 * tm;
            uint32_t* dst = reinterpret_cast<uint32_t*>(base + m * a.c_sm);
#pragma unroll
            for (int ob = 0; ob < GN; ++ob) {
                const floatx4 t0 = acc[tm][2 * ob], t1 = acc[tm][2 * ob + 1];
                const auto s0 = __builtin_amdgcn_permlane16_swap(pack2<T>(t0[0], t0[1]), pack2<T>(t1[0], t1[1]), false, false);
                const auto s1 = __builtin_amdgcn_permlane16_swap(pack2<T>(t0[2], t0[3]), pack2<T>(t1[2], t1[3]), false, false);
                if (m < a.M) __builtin_nontemporal_store(uintx4{s0[0], s1[0], s0[1], s1[1]}, reinterpret_cast<uintx4*>(dst + 16 * ob));
            }
            reset(tm);
        }
    };
    if (nin == 0) {                                         // no input block: zero rows
        for (int tile = 0; tile < n_tiles; ++tile) store_tile(tile);
        return;
    }

    const int npair = (nin + 1) / 2, n_steps = n_tiles * npair;
    // weights: the wave's transfers of 16 rows (1 KB) of a step's 4 GN half blocks
    const uint32_t wlane = (uint32_t)((lane >> 2) * 64 + 16 * ((lane & 3) ^ (lane >> 4)));
    const int32_t* wlist[2];
    int whf[2], wdst[2], whalf[2], wblk[2];
    bool wlive[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int u = w + 8 * j, hf = u >= NT, rem = u - NT * hf;
        wlive[j] = u < 2 * NT;
        whf[j] = hf;
        whalf[j] = (rem & 1) * 1024;
        wdst[j] = hf * 8192 + rem * 1024;
        wlist[j] = a.seg_blk + (wlive[j] ? a.seg_ptr[row0 + (rem >> 1)] : p0);
        wblk[j] = table_entry(wlist[j] + min(hf, nin - 1));
    }
    int w_t = 0;                                            // weight cursor: pair of entries inside the tile
    auto transfer_w = [&](int buf) __attribute__((always_inline)) {
        if (++w_t == npair) w_t = 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (wlive[j]) dma_to_lds_at(spz + (long)wblk[j] * 2048 + whalf[j], wlane, lds + buf * 16384 + wdst[j]);
            wblk[j] = table_entry(wlist[j] + min(2 * w_t + whf[j], nin - 1));       // (an odd list's last step: the last entry twice)
        }
    };
    // activations, as in bs_dds32d_kernel: chunk 4 hf + c of token t lies at chunk (4 hf + c) ^ ((t >> 1) & 7)
    char* stage = lds + 32768 + 8192 * w;                   // the second stage 64 KB behind the first
    const int tl = lane >> 3;
    uint32_t xoff[NX];
#pragma unroll
    for (int j = 0; j < NX; ++j) xoff[j] = 0;
    int f_tile = 0, f_t = 0;                                // transfer cursor: (token tile, pair of entries inside it)
    int in0 = table_entry(a.seg_inner + p0), in1 = table_entry(a.seg_inner + p0 + min(1, nin - 1));
    uint32_t xeven = 0, xodd = 0;
    auto transfer_head = [&]() __attribute__((always_inline)) {
        if (f_t == 0) {
            const long m0 = ((long)ty + (long)f_tile * gy) * 512 + 64 * w;
#pragma unroll
            for (int j = 0; j < NX; ++j) {
                const int t = 8 * j + tl, c = (lane & 7) ^ ((t >> 1) & 7);
                const long m = min(m0 + t, (long)a.M - 1);   // clamped: masked at the store (past the last tile: never read)
                xoff[j] = (uint32_t)((m * a.dn_sm + 8 * (c & 3)) * 2);
            }
        }
        const uint32_t b0 = (uint32_t)in0 * 64u, b1 = (uint32_t)in1 * 64u;
        const bool second = (((lane & 7) ^ (tl >> 1)) >> 2) != 0;             // even j: which of the two blocks the lane's chunk belongs to
        xeven = second ? b1 : b0;
        xodd = second ? b0 : b1;
        if (++f_t == npair) { f_t = 0; ++f_tile; }
        in0 = table_entry(a.seg_inner + p0 + 2 * f_t);
        in1 = table_entry(a.seg_inner + p0 + min(2 * f_t + 1, nin - 1));
    };
    auto transfer_row = [&](int st, int j) __attribute__((always_inline)) {
        dma_to_lds_at(xb, xoff[j] + ((j & 1) ? xodd : xeven), stage + 65536 * st + 1024 * j);
    };
    int xfrag[2][TM];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int t = 16 * tm + r16;
            xfrag[hf][tm] = t * 128 + 16 * ((4 * hf + g) ^ ((t >> 1) & 7));
        }
    // the row operand of tile 2 ob + h of an entry: outputs 16 h + r16, contraction slots 8 g .. 8 g + 7
    int wfrag[WT ? 4 : 1];
    if (WT) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                const int row = 8 * g + 4 * part + (r16 >> 2), c = 2 * h + ((r16 & 3) >> 1);
                wfrag[WT ? 2 * h + part : 0] = row * 64 + 16 * (c ^ ((row >> 2) & 3)) + 8 * (r16 & 1);
            }
    } else wfrag[0] = r16 * 64 + 16 * (g ^ (r16 >> 2));

    transfer_w(0);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
        transfer_head();
#pragma unroll
        for (int j = 0; j < NX; ++j) transfer_row(st, j);
    }
    int c_tile = 0, c_t = 0;                                // compute cursor: tile, step inside it
    for (int step = 0; step < n_steps; ++step) {
        const int cur = step & 1;
        drain_loads_but<NX>();                              // all but the next step's activations (stores of a tile wait too)
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();                       // the step's weights are there, the other buffer is free
        asm volatile("" ::: "memory");
        transfer_w(cur ^ 1);                                // (the last step's are not used)
        uintx4 fx[2][TM];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) fx[hf][tm] = *reinterpret_cast<const uintx4*>(stage + 65536 * cur + xfrag[hf][tm]);
        __builtin_amdgcn_s_waitcnt(0xC07F);                 // lgkmcnt(0): the fragments are in registers, the stage is free
        transfer_head();
        // the transfers of step + 2 go out between the products: eight waves that ask for everything behind the barrier wait in
        // line with idle matrix cores
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            if (2 * c_t + hf < nin) {                       // workgroup-uniform
                const char* wb = lds + 16384 * cur + hf * 8192;
                uintx4 fw[2];
                auto weights = [&](int n) __attribute__((always_inline)) {
                    const char* p = wb + (n >> 1) * 2048;
                    if (WT) fw[n & 1] = lds_read_tr8(p + wfrag[WT ? 2 * (n & 1) : 0], p + wfrag[WT ? 2 * (n & 1) + 1 : 0]);
                    else fw[n & 1] = *reinterpret_cast<const uintx4*>(p + (n & 1) * 1024 + wfrag[0]);
                };
                weights(0);
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    if (n + 1 < NT) weights(n + 1);
                    __builtin_amdgcn_sched_barrier(0x47f);  // (reads stay in front of the products before those that need them)
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
                        acc[tm][n] = Frag32<T>::mma(__builtin_bit_cast(uint4, fw[n & 1]), __builtin_bit_cast(uint4, fx[hf][tm]), acc[tm][n]);
#pragma unroll
                    for (int j = 0; j < TM; ++j)
                        if (j * NT / TM == n) transfer_row(cur, TM * hf + j);
                    __builtin_amdgcn_sched_barrier(0x47f);
                }
            } else {
#pragma unroll
                for (int j = 0; j < TM; ++j) transfer_row(cur, TM * hf + j);
            }
        }
        if (++c_t == npair) { store_tile(c_tile); c_t = 0; ++c_tile; }
    }
    drain_loads();                                          // (transfers past the last step)
}

template <typename T, bool WT>
__global__ __launch_bounds__(512) void bs_dds32c_kernel(DdsGroupArgs a, int n_streams) {
    extern __shared__ __attribute__((aligned(1024))) uint16_t wres[];   // 2 x [entry][output block][row][32], then 2 x 8 stages of 8 KB
    char* lds = reinterpret_cast<char*>(wres);
    const int per_xcd = (int)gridDim.x / a.n_xcd;
    const int pair = ((int)blockIdx.x % a.n_xcd) * per_xcd + (int)blockIdx.x / a.n_xcd;
    if (pair >= n_streams * a.n_grp) return;                // workgroup-uniform
    const int ty = pair / a.n_grp, grp = pair % a.n_grp;
    if (ty >= (a.M + 511) / 512) return;
    switch (a.grp_n[grp]) {
        case 4: dds32c_group<T, WT, 4>(a, lds, grp, ty, n_streams); break;
        case 3: dds32c_group<T, WT, 3>(a, lds, grp, ty, n_streams); break;
        case 2: dds32c_group<T, WT, 2>(a, lds, grp, ty, n_streams); break;
        default: dds32c_group<T, WT, 1>(a, lds, grp, ty, n_streams); break;
    }
}

// ---------------------------------------------------------------------------------------
// fused block-sparse attention: out = softmax(scale * Q K^T + key mask) V over the nonzero blocks
// ---------------------------------------------------------------------------------------
// One pass for 32x32 blocks of a 2-byte type: the (Z, nnz, 32, 32) score and probability tensors of
// the SDD -> softmax -> DSD sequence never exist.  One workgroup per (batch, head, NW consecutive
// block-rows); wave w owns the 32 queries of block-row NW*group + w with their Q fragments in
// registers.  The workgroup walks the union of the rows' column lists; each step stages one 32 x D
// tile of K (row-major) and of V (transposed, [d][key slot]) in LDS, double-buffered, and every
// wave whose row holds that column forms S^T = K Q^T (rows = keys, columns = queries: a lane then
// owns one query per 16-column tile and its row statistics are lane scalars plus a 4-group
// butterfly), runs the online softmax in base 2, and accumulates O^T += V^T P with the
// probabilities going straight from the score registers into the MFMA operand: key 16kt + 4g + i
// sits in contraction slot 8g + 4kt + i, which is the order the V tile is transposed into.
struct AttnArgs {
    const void* q; const void* k; const void* v; void* out;
    const int32_t* uni_ptr; const int32_t* uni_inner; const int32_t* uni_blk;
    const float* kpm; long kpm_stride;
    int brows_per_head, grps_per_head, n_heads, Z;
    long q_sz, q_sh, q_sm, k_sz, k_sh, k_sn, v_sz, v_sh, v_sn, o_sz, o_sh, o_sm;
    float scale;
    float* lse2;        // optional (Z, H, 32 * brows_per_head): base-2 log of every row's softmax denominator
    int n_xcd;          // dies the dispatcher deals workgroup ids to (set where the kernel is launched)
    const float* am; long am_stride;     // optional (rows, cols) additive term per (query, key), shared by batch and heads
    // dropout of the probabilities (DROP kernels): element (z, head, query, key) is kept when the hash of
    // (seed, row = (z H + head) L + query, key) reaches the threshold; kept ones are scaled by 1 / (1 - p)
    uint32_t drop_seed, drop_thresh; float drop_scale;
};

// Maxima of scores.  A two-operand fmaxf costs three instructions here (each operand is first quieted
// by a self-maximum); three-operand maxima are emitted as they are, so pairs get -inf as a third.
__device__ __forceinline__ float max2_finite(float a, float b) { return fmaxf(fmaxf(a, b), -INFINITY); }
__device__ __forceinline__ float max8_finite(floatx4 a, floatx4 b) {
    const float m0 = fmaxf(fmaxf(a[0], a[1]), a[2]);
    const float m1 = fmaxf(fmaxf(m0, a[3]), b[0]);
    const float m2 = fmaxf(fmaxf(m1, b[1]), b[2]);
    return max2_finite(m2, b[3]);
}
__device__ __forceinline__ float group_max_finite(float v) {
    float a, b;
    rows_pair16(v, a, b); v = max2_finite(a, b);
    rows_pair32(v, a, b); return max2_finite(a, b);
}

// LDS image of a block-column's K and V tiles: rows of 2 D bytes without padding (a wave's direct-to-LDS load
// fills 1024 consecutive bytes), 16-byte chunks permuted within a row so that the fragment reads spread over the
// banks: the eight lanes of a 16-byte K read (eight consecutive keys, one chunk) and the sixteen lanes of a
// transposing V read (four consecutive keys, 32 bytes each) then cover a 128-byte line exactly.  Both maps are
// their own inverses.  CPR = chunks per row.
template <int CPR> __device__ __forceinline__ int attn_kslot(int row, int c) {
    constexpr int RPL = CPR >= 8 ? 1 : 8 / CPR;           // rows per 128-byte line
    return c ^ ((row / RPL) & (CPR - 1));
}
template <int CPR> __device__ __forceinline__ int attn_vslot(int row, int c) {
    constexpr int RPL = CPR >= 8 ? 1 : 8 / CPR;
    return c ^ ((((row / RPL) & 3) & (CPR / 2 - 1)) << 1);
}
template <typename T, int KS, int NW, bool MASKED, bool DROP = false>     // head dim 32*KS, NW block-rows (waves) per workgroup
__global__ __launch_bounds__(64 * NW) void bs_attn32_kernel(const AttnArgs a) {
    constexpr int D = 32 * KS, DT = D / 16, RB = 2 * D;   // RB: bytes of a tile row
    // block-columns per step: what 64 KB of LDS hold twice over -- half of that for workgroups of four waves at 64 dims,
    // of which a compute unit then holds four (the registers allow it) instead of two
    constexpr int CP = KS == 1 ? 4 : (KS == 2 && NW >= 8 ? 4 : 2);
    constexpr int CPR = D / 8;                            // 16-byte chunks per tile row
    constexpr int COLB = 64 * RB;                         // one column's image: rows 0..31 keys of K, 32..63 the same keys of V
    constexpr int U = COLB / 1024, NCH = (U + NW - 1) / NW;      // wave loads per column, and per wave
    constexpr float LOG2E = 1.4426950408889634f;
    // The running reference exponent of a query is only raised (and its accumulators rescaled) when
    // a block's maximum exceeds it by more than LAZY binary orders of magnitude; until then the
    // probabilities may exceed 1 (by at most 2^LAZY), which fp32 sums and 2-byte operands hold
    // without loss, and the result is the same quotient.
    constexpr float LAZY = 8.f;
    __shared__ __attribute__((aligned(1024))) char tiles[2][CP][COLB];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int unit, grp;
    if (!unit_of(blockIdx.x, a.n_xcd, a.grps_per_head, a.n_heads * a.Z, unit, grp)) return;
    const int z = unit / a.n_heads, head = unit % a.n_heads;
    const int ug = head * a.grps_per_head + grp;
    const int p0 = a.uni_ptr[ug], n = a.uni_ptr[ug + 1] - p0;
    const int bi = grp * NW + w;
    const bool have_row = bi < a.brows_per_head;
    const T* qp = reinterpret_cast<const T*>(a.q) + z * a.q_sz + head * a.q_sh +
                  (long)(min(bi, a.brows_per_head - 1) * 32 + r16) * a.q_sm + 8 * g;
    const T* kz = reinterpret_cast<const T*>(a.k) + z * a.k_sz + head * a.k_sh;
    const T* vz = reinterpret_cast<const T*>(a.v) + z * a.v_sz + head * a.v_sh;
    const float* kpm = a.kpm ? a.kpm + z * a.kpm_stride : nullptr;

    uintx4 fq[2][KS];                                     // B operand: query 16qt + r16, dims 32ks + 8g ..
#pragma unroll
    for (int qt = 0; qt < 2; ++qt)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fq[qt][ks] = *reinterpret_cast<const uintx4*>(qp + 16 * qt * a.q_sm + 32 * ks);

    // staging: wave load x = w + NW i of a column fills bytes 1024 x .. of its image; this lane's 16 of them are
    // chunk slot `p` of image row `row`
    const T* src[NCH];           // the lane's chunk in block-column 0
    long src_step[NCH];          // elements from one block-column to the next (wave-uniform)
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int pos = 1024 * (w + NW * i) + 16 * lane, row = (pos / RB) & 63, p = (pos % RB) / 16;
        const bool is_k = 1024 * (w + NW * i) < 32 * RB;    // whole wave loads are K or V
        src[i] = is_k ? kz + (long)row * a.k_sn + 8 * attn_kslot<CPR>(row, p)
                      : vz + (long)(row - 32) * a.v_sn + 8 * attn_vslot<CPR>(row - 32, p);
        src_step[i] = is_k ? 32 * a.k_sn : 32 * a.v_sn;
    }
    auto fetch = [&](int j, int stage, int inner) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NCH; ++i)
            if (U % NW == 0 || w + NW * i < U) dma_to_lds(src[i] + inner * src_step[i], tiles[stage][j] + 1024 * (w + NW * i));
    };

    floatx4 o[DT][2];                                     // O^T[d = 16dt + 4g + i][query 16qt + r16]
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) { o[dt][0] = Frag<float>::zero(); o[dt][1] = Frag<float>::zero(); }
    float m_run[2] = {-INFINITY, -INFINITY};
    floatx4 lsum[2] = {Frag<float>::zero(), Frag<float>::zero()};      // every element: sum of the query's probabilities
    const uint32_t one2 = pack2<T>(1.f, 1.f);
    const uintx4 ones = {one2, one2, one2, one2};
    const float scale2 = a.scale * LOG2E;

    // S^T[key 16kt + 4g + i][query 16qt + r16] of the K tile at `tile`
    floatx4 sc[2][2];
    floatx4 amk[2][2];                                    // the attention-mask entries of sc (asked for with the scores)
    const float* amrow = (MASKED && a.am) ? a.am + (long)(min(bi, a.brows_per_head - 1) * 32 + r16) * a.am_stride + 4 * g : nullptr;
    uint32_t drop_row[2] = {0u, 0u};                      // DROP: hash of (seed, global row) of the lane's two queries
    if (DROP) {
        const uint32_t row0 = (uint32_t)(z * a.n_heads + head) * (uint32_t)(a.brows_per_head * 32) +
                              (uint32_t)(min(bi, a.brows_per_head - 1) * 32 + r16);
        drop_row[0] = drop_row_hash(a.drop_seed, row0);
        drop_row[1] = drop_row_hash(a.drop_seed, row0 + 16u);
    }
    auto score = [&](const char* tile, int inner) __attribute__((always_inline)) {
        if (MASKED && amrow) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int qt = 0; qt < 2; ++qt)
                    amk[kt][qt] = *reinterpret_cast<const floatx4*>(amrow + 16 * qt * a.am_stride + (long)inner * 32 + 16 * kt);
        }
        uintx4 fk[2][KS];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                fk[kt][ks] = *reinterpret_cast<const uintx4*>(tile + (16 * kt + r16) * RB + 16 * attn_kslot<CPR>(16 * kt + r16, 4 * ks + g));
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                sc[kt][qt] = Frag<float>::zero();
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) sc[kt][qt] = mma32<T>(fk[kt][ks], fq[qt][ks], sc[kt][qt]);
            }
    };
    // DROP: the probabilities that go to the product with V, the dropped ones zeroed (the denominator sums all of them).  A
    // packed pair is a pair of columns with one hash: three 16-bit vector instructions instead of a compare, a select and a
    // second rounding per element
    auto dropped = [&](uintx4 p, uint32_t row_hash, int inner) __attribute__((always_inline)) {
        const uint32_t pair0 = (uint32_t)inner * 16u + 2u * g;
#pragma unroll
        for (int i = 0; i < 4; ++i)                       // columns 4 g + 2 (i & 1) + 16 (i >> 1)
            p[i] = drop_packed(p[i], drop_mix(row_hash + (pair0 + (i & 1) + 8u * (i >> 1)) * 0x632BE5ABu), a.drop_thresh);
        return p;
    };
    // online softmax of sc and O^T += V^T P with the V tile that follows the K tile at `tile`; `inner` = its block-column
    auto soft_pv = [&](const char* tile, int inner) __attribute__((always_inline)) {
        // A operand: column d = 16dt + r16 of V, keys 4g .. 4g+3 and 16+4g .. 16+4g+3
        const int vrow = 4 * g + (r16 >> 2);
        const char* vp = tile + (32 + vrow) * RB + 8 * (r16 & 1);
        uintx4 fv[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const char* p0 = vp + 16 * attn_vslot<CPR>(vrow, 2 * dt + ((r16 & 3) >> 1));
            fv[dt] = lds_read_tr8(p0, p0 + 16 * RB);
        }
        uintx4 pb[2], pd[2];                              // probabilities, and (DROP) the kept ones
        if (!MASKED) {
            // scale > 0 and no mask: the maximum is taken on the raw scores and the scale rides in
            // the exponent's fma
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                const floatx4 s0 = sc[0][qt], s1 = sc[1][qt];
                const float mx = group_max_finite(max8_finite(s0, s1)) * scale2;
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(mx > m_run[qt] + LAZY) != 0, 0)) {      // wave-uniform: some row maximum grew a lot
                    asm volatile("");                        // (stays a branch: the compiler would do the multiplications always)
                    const float m_new = fmaxf(m_run[qt], mx);
                    const float alpha = __builtin_amdgcn_exp2f(m_run[qt] - m_new);
                    m_run[qt] = m_new;
                    lsum[qt] *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[dt][qt] *= alpha;
                }
                const float nm = -m_run[qt];
                float e0[4], e1[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    e0[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[i], scale2, nm));
                    e1[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s1[i], scale2, nm));
                }
                pb[qt] = uintx4{pack2<T>(e0[0], e0[1]), pack2<T>(e0[2], e0[3]), pack2<T>(e1[0], e1[1]), pack2<T>(e1[2], e1[3])};
                if (DROP) pd[qt] = dropped(pb[qt], drop_row[qt], inner);
            }
        } else {
            floatx4 mk[2] = {Frag<float>::zero(), Frag<float>::zero()};
            if (kpm) {
                const float* mp = kpm + (long)inner * 32 + 4 * g;
                mk[0] = *reinterpret_cast<const floatx4*>(mp) * LOG2E;
                mk[1] = *reinterpret_cast<const floatx4*>(mp + 16) * LOG2E;
            }
#pragma unroll
            for (int qt = 0; qt < 2; ++qt) {
                floatx4 t0 = sc[0][qt] * scale2 + mk[0], t1 = sc[1][qt] * scale2 + mk[1];
                if (amrow) { t0 += amk[0][qt] * LOG2E; t1 += amk[1][qt] * LOG2E; }
                float mx = fmaxf(fmaxf(fmaxf(t0[0], t0[1]), t0[2]), fmaxf(fmaxf(t0[3], t1[0]), t1[1]));
                mx = fmaxf(fmaxf(mx, t1[2]), t1[3]);
                mx = group_max(mx);
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(mx > m_run[qt] + LAZY) != 0, 0)) {
                    asm volatile("");
                    const float m_new = fmaxf(m_run[qt], mx);
                    const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m_run[qt] - m_new);
                    m_run[qt] = m_new;
                    lsum[qt] *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[dt][qt] *= alpha;
                }
                const float mref = (m_run[qt] == -INFINITY) ? 0.f : m_run[qt];     // all keys masked so far: p = 0
                float e0[4], e1[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    e0[i] = __builtin_amdgcn_exp2f(t0[i] - mref);
                    e1[i] = __builtin_amdgcn_exp2f(t1[i] - mref);
                }
                pb[qt] = uintx4{pack2<T>(e0[0], e0[1]), pack2<T>(e0[2], e0[3]), pack2<T>(e1[0], e1[1]), pack2<T>(e1[2], e1[3])};
                if (DROP) pd[qt] = dropped(pb[qt], drop_row[qt], inner);
            }
        }
        // the row sums come from the matrix pipe as well: a row of ones times the rounded probabilities
        lsum[0] = mma32<T>(ones, pb[0], lsum[0]);
        lsum[1] = mma32<T>(ones, pb[1], lsum[1]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            o[dt][0] = mma32<T>(fv[dt], DROP ? pd[0] : pb[0], o[dt][0]);
            o[dt][1] = mma32<T>(fv[dt], DROP ? pd[1] : pb[1], o[dt][1]);
        }
    };

    // The index lists are read two steps (block-column) and one step (presence) ahead of their use,
    // so that no step waits for a table load.  A step: ask for the next step's tiles (they go into the
    // other stage, which every wave has finished reading before the last barrier), work through this
    // step's columns, wait for the own loads, barrier.
    const int n_steps = (n + CP - 1) / CP;
    int inner_cur[CP], inner_n1[CP], blk_cur[CP];
#pragma unroll
    for (int j = 0; j < CP; ++j) {
        inner_cur[j] = j < n ? table_entry(a.uni_inner + p0 + j) : 0;
        inner_n1[j] = CP + j < n ? table_entry(a.uni_inner + p0 + CP + j) : 0;
        blk_cur[j] = j < n ? table_entry(a.uni_blk + (long)(p0 + j) * NW + w) : -1;
    }
    if (n > 0) {
#pragma unroll
        for (int j = 0; j < CP; ++j)
            if (j < n) fetch(j, 0, inner_cur[j]);
    }
    drain_loads();
    __syncthreads();
    for (int st = 0; st < n_steps; ++st) {
        const int s1 = CP * (st + 1), s2 = CP * (st + 2);
        int inner_n2[CP], blk_n1[CP];
#pragma unroll
        for (int j = 0; j < CP; ++j) {
            inner_n2[j] = s2 + j < n ? table_entry(a.uni_inner + p0 + s2 + j) : 0;
            blk_n1[j] = s1 + j < n ? table_entry(a.uni_blk + (long)(p0 + s1 + j) * NW + w) : -1;
        }
#pragma unroll
        for (int j = 0; j < CP; ++j)
            if (s1 + j < n) fetch(j, (st + 1) & 1, inner_n1[j]);
#pragma unroll
        for (int j = 0; j < CP; ++j) {
            if (have_row && blk_cur[j] >= 0) {
                score(tiles[st & 1][j], inner_cur[j]);
                soft_pv(tiles[st & 1][j], inner_cur[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < CP; ++j) {
            inner_cur[j] = inner_n1[j];
            inner_n1[j] = inner_n2[j];
            blk_cur[j] = blk_n1[j];
        }
        drain_loads();                                    // this wave's part of the next step's tiles has landed
        __syncthreads();
    }
    if (!have_row) return;
    T* op = reinterpret_cast<T*>(a.out) + z * a.o_sz + head * a.o_sh;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
        const float l = lsum[qt][0];
        float inv = l > 0.f ? 1.0f / l : 0.f;             // rows without a finite score come out as zeros
        if (DROP) inv *= a.drop_scale;
        T* row = op + ((long)bi * 32 + 16 * qt + r16) * a.o_sm + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) store4_f32(row + 16 * dt, o[dt][qt] * inv);
        if (a.lse2 && g == 0)       // a row without a finite score: +inf, so that 2^(score - lse2) is 0
            a.lse2[(((long)z * a.n_heads + head) * a.brows_per_head + bi) * 32 + 16 * qt + r16] =
                l > 0.f ? m_run[qt] + __log2f(l) : INFINITY;
    }
}

// ---------------------------------------------------------------------------------------
// row operations: one wave per row of a block-row
// ---------------------------------------------------------------------------------------
struct RowArgs {
    void* x; void* out;
    const int32_t* row_ptr; const int32_t* row_blk; const int32_t* row_col;
    int n_brow, brows_per_head, blk_shift;
    long x_sz;
    float scale;
    const float* kpm; long kpm_stride; int kpm_mul;
    const float* am; long am_stride; int am_mul;
    int op;
};

__device__ __forceinline__ float mask_term(float v, int mul) {
    if (!mul) return v;
    return v == 0.f ? -INFINITY : 0.f;
}

// value of element e (0 <= e < nb*blk) of the row, with scale and masks applied
template <typename T>
__device__ __forceinline__ float row_value(const RowArgs& a, const T* xz, int p0, int rl, int e, int z, int grow,
                                           long* addr) {
    const int BLK = 1 << a.blk_shift;
    const int bidx = e >> a.blk_shift, cl = e & (BLK - 1);
    const long off = (long)a.row_blk[p0 + bidx] * (BLK * BLK) + rl * BLK + cl;
    *addr = off;
    float v = Elem<T>::to_f32(xz[off]) * a.scale;
    if (a.kpm || a.am) {
        const long col = (long)a.row_col[p0 + bidx] * BLK + cl;
        if (a.kpm) v += mask_term(a.kpm[z * a.kpm_stride + col], a.kpm_mul);
        if (a.am) v += mask_term(a.am[grow * a.am_stride + col], a.am_mul);
    }
    return v;
}

template <typename T, int NREG>
__global__ __launch_bounds__(256) void bs_softmax_kernel(RowArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int BLK = 1 << a.blk_shift;
    const long R = (long)blockIdx.x * 4 + w;
    if (R >= (long)a.n_brow * BLK) return;
    const int brow = (int)(R >> a.blk_shift), rl = (int)(R & (BLK - 1));
    const int z = blockIdx.y;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const int n = nb << a.blk_shift;
    const int grow = (brow % a.brows_per_head) * BLK + rl;
    T* xz = reinterpret_cast<T*>(a.x) + z * a.x_sz;

    float vals[NREG];
    long addr[NREG];
    float mx = -INFINITY;
#pragma unroll
    for (int it = 0; it < NREG; ++it) {
        const int e = lane + 64 * it;
        vals[it] = -INFINITY;
        addr[it] = 0;
        if (e < n) vals[it] = row_value<T>(a, xz, p0, rl, e, z, grow, &addr[it]);
        mx = fmaxf(mx, vals[it]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int it = 0; it < NREG; ++it) {
        const int e = lane + 64 * it;
        if (e < n) { vals[it] = expf(vals[it] - mx); sum += vals[it]; }   // -inf - -inf = NaN, kept on purpose
    }
    sum = wave_sum(sum);
    const float inv = 1.0f / sum;
#pragma unroll
    for (int it = 0; it < NREG; ++it) {
        const int e = lane + 64 * it;
        if (e < n) xz[addr[it]] = Elem<T>::from_f32(vals[it] * inv);
    }
}

// Fast path for 32x32 blocks of a 2-byte type: one workgroup per (block-row, 16-row half).  The
// 16 x 32 half of a block is 1 KiB of contiguous memory, which one wave moves with a single 16-byte
// load per lane (lane = 4*row + chunk of 8 columns); wave w owns blocks w, w+4, ... of the row and
// keeps them in registers (raw 2-byte form) across the max / sum / write passes, so HBM sees each
// element once in and once out.  Row statistics go quad -> wave (DPP) -> workgroup (LDS).
template <typename T, int MAXB, int NW>     // NW waves share a (block-row, 16-row half); wave w takes blocks w, w + NW, ...
__global__ __launch_bounds__(64 * NW) void bs_softmax32_kernel(RowArgs a) {
    constexpr float LOG2E = 1.4426950408889634f;
    __shared__ float red[2][NW][16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, rl = lane >> 2, chunk = lane & 3;
    const int brow = blockIdx.x >> 1, row = (blockIdx.x & 1) * 16 + rl;       // row inside the block
    const int z = blockIdx.y;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const int grow = (brow % a.brows_per_head) * 32 + row;
    T* xz = reinterpret_cast<T*>(a.x) + z * a.x_sz + row * 32 + chunk * 8;
    const bool masked = a.kpm || a.am;

    uint4 raw[MAXB];
    long off[MAXB];
#pragma unroll
    for (int it = 0; it < MAXB; ++it) {
        const int j = w + NW * it;
        off[it] = -1;
        if (j < nb) {
            off[it] = (long)a.row_blk[p0 + j] * 1024;
            // streamed once in, once out: nontemporal both ways
            const uintx4 t_ = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(xz + off[it]));
            raw[it] = make_uint4(t_[0], t_[1], t_[2], t_[3]);
        }
    }
    // element u (0..7) of block slot `it` as float, unscaled
    auto elem = [&](int it, int u) -> float {
        const uint32_t word = (&raw[it].x)[u >> 1];
        T e;
        *reinterpret_cast<uint16_t*>(&e) = (u & 1) ? (uint16_t)(word >> 16) : (uint16_t)(word & 0xffffu);
        return Elem<T>::to_f32(e);
    };
    // additive mask term of that element (masked launches only)
    auto mask_of = [&](int it, int u) -> float {
        const long col = (long)a.row_col[p0 + w + NW * it] * 32 + chunk * 8 + u;
        float v = 0.f;
        if (a.kpm) v += mask_term(a.kpm[z * a.kpm_stride + col], a.kpm_mul);
        if (a.am) v += mask_term(a.am[grow * a.am_stride + col], a.am_mul);
        return v;
    };
    // pass 1: row maximum of x*scale (+ masks)
    float mx = -INFINITY;
    if (!masked && a.scale > 0.f) {              // max commutes with a positive scale: one multiply per lane
#pragma unroll
        for (int it = 0; it < MAXB; ++it)
            if (off[it] >= 0)
#pragma unroll
                for (int u = 0; u < 8; ++u) mx = fmaxf(mx, elem(it, u));
        mx *= a.scale;
    } else {
#pragma unroll
        for (int it = 0; it < MAXB; ++it)
            if (off[it] >= 0)
#pragma unroll
                for (int u = 0; u < 8; ++u) mx = fmaxf(mx, elem(it, u) * a.scale + (masked ? mask_of(it, u) : 0.f));
    }
    mx = fmaxf(mx, __shfl_xor(mx, 1));
    mx = fmaxf(mx, __shfl_xor(mx, 2));
    if (chunk == 0) red[0][w][rl] = mx;
    __syncthreads();
    mx = red[0][0][rl];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) mx = fmaxf(mx, red[0][ww][rl]);
    // pass 2: exponentials (kept as floats in registers) and their sum; -inf - -inf = NaN, kept
    const float mx2 = mx * LOG2E, scale2 = a.scale * LOG2E;
    float ev[MAXB][8];
    float sum = 0.f;
#pragma unroll
    for (int it = 0; it < MAXB; ++it)
        if (off[it] >= 0)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                float arg = elem(it, u) * scale2 - mx2;
                if (masked) arg += mask_of(it, u) * LOG2E;
                ev[it][u] = __builtin_amdgcn_exp2f(arg);
                sum += ev[it][u];
            }
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if (chunk == 0) red[1][w][rl] = sum;
    __syncthreads();
    sum = red[1][0][rl];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) sum += red[1][ww][rl];
    const float inv = 1.0f / sum;
    // pass 3: normalise, round once, store
#pragma unroll
    for (int it = 0; it < MAXB; ++it)
        if (off[it] >= 0) {
            uint32_t outw[4];
#pragma unroll
            for (int u2 = 0; u2 < 4; ++u2) {
                T lo = Elem<T>::from_f32(ev[it][2 * u2] * inv);
                T hi = Elem<T>::from_f32(ev[it][2 * u2 + 1] * inv);
                outw[u2] = (uint32_t)*reinterpret_cast<uint16_t*>(&lo) | ((uint32_t)*reinterpret_cast<uint16_t*>(&hi) << 16);
            }
            __builtin_nontemporal_store(uintx4{outw[0], outw[1], outw[2], outw[3]}, reinterpret_cast<uintx4*>(xz + off[it]));
        }
}

// Backward of the block softmax for 32x32 blocks of a 2-byte type, one pass: dx = scale * y * (dy - sum_row(dy * y)).
// Same work split as bs_softmax32_kernel (workgroup per (block-row, 16-row half), wave w takes blocks
// w, w+NW, ...; a lane holds 8 consecutive elements of one row per block): y and dy stay in registers
// in their 2-byte form between the row sum and the result, so HBM sees two reads and one write.
struct RowBwdArgs {
    const void* y; const void* dy; void* dx;
    const int32_t* row_ptr; const int32_t* row_blk;
    long y_sz;
    float scale;
};

template <typename T, int MAXB, int NW>
__global__ __launch_bounds__(64 * NW) void bs_softmax32_bwd_kernel(RowBwdArgs a) {
    __shared__ float red[NW][16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, rl = lane >> 2, chunk = lane & 3;
    const int brow = blockIdx.x >> 1, row = (blockIdx.x & 1) * 16 + rl;
    const int z = blockIdx.y;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const long base = z * a.y_sz + row * 32 + chunk * 8;
    const T* yz = reinterpret_cast<const T*>(a.y) + base;
    const T* dz = reinterpret_cast<const T*>(a.dy) + base;
    T* xz = reinterpret_cast<T*>(a.dx) + base;

    uintx4 ry[MAXB], rd[MAXB];
    int blk[MAXB];
#pragma unroll
    for (int it = 0; it < MAXB; ++it) {
        const int j = w + NW * it;
        blk[it] = -1;
        if (j < nb) {
            blk[it] = a.row_blk[p0 + j];
            ry[it] = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(yz + (long)blk[it] * 1024));
            rd[it] = __builtin_nontemporal_load(reinterpret_cast<const uintx4*>(dz + (long)blk[it] * 1024));
        }
    }
    auto elem = [&](uint32_t word, int hi) -> float {
        T e;
        *reinterpret_cast<uint16_t*>(&e) = hi ? (uint16_t)(word >> 16) : (uint16_t)(word & 0xffffu);
        return Elem<T>::to_f32(e);
    };
    float s = 0.f;
#pragma unroll
    for (int it = 0; it < MAXB; ++it)
        if (blk[it] >= 0)
#pragma unroll
            for (int u = 0; u < 8; ++u) s += elem(ry[it][u >> 1], u & 1) * elem(rd[it][u >> 1], u & 1);
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (chunk == 0) red[w][rl] = s;
    __syncthreads();
    s = red[0][rl];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) s += red[ww][rl];
#pragma unroll
    for (int it = 0; it < MAXB; ++it)
        if (blk[it] >= 0) {
            uint32_t outw[4];
#pragma unroll
            for (int u2 = 0; u2 < 4; ++u2) {
                const float lo = a.scale * elem(ry[it][u2], 0) * (elem(rd[it][u2], 0) - s);
                const float hi = a.scale * elem(ry[it][u2], 1) * (elem(rd[it][u2], 1) - s);
                outw[u2] = pack2<T>(lo, hi);
            }
            __builtin_nontemporal_store(uintx4{outw[0], outw[1], outw[2], outw[3]},
                                        reinterpret_cast<uintx4*>(xz + (long)blk[it] * 1024));
        }
}

// rows longer than the register budget: three passes over the row
template <typename T>
__global__ __launch_bounds__(256) void bs_softmax_long_kernel(RowArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int BLK = 1 << a.blk_shift;
    const long R = (long)blockIdx.x * 4 + w;
    if (R >= (long)a.n_brow * BLK) return;
    const int brow = (int)(R >> a.blk_shift), rl = (int)(R & (BLK - 1));
    const int z = blockIdx.y;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const int n = nb << a.blk_shift;
    const int grow = (brow % a.brows_per_head) * BLK + rl;
    T* xz = reinterpret_cast<T*>(a.x) + z * a.x_sz;
    long addr;
    float mx = -INFINITY;
    for (int e = lane; e < n; e += 64) mx = fmaxf(mx, row_value<T>(a, xz, p0, rl, e, z, grow, &addr));
    mx = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < n; e += 64) sum += expf(row_value<T>(a, xz, p0, rl, e, z, grow, &addr) - mx);
    sum = wave_sum(sum);
    const float inv = 1.0f / sum;
    for (int e = lane; e < n; e += 64) {
        const float v = expf(row_value<T>(a, xz, p0, rl, e, z, grow, &addr) - mx) * inv;
        xz[addr] = Elem<T>::from_f32(v);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void bs_rowreduce_kernel(RowArgs a) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int BLK = 1 << a.blk_shift;
    const long R = (long)blockIdx.x * 4 + w;
    if (R >= (long)a.n_brow * BLK) return;
    const int brow = (int)(R >> a.blk_shift), rl = (int)(R & (BLK - 1));
    const int z = blockIdx.y;
    const int p0 = a.row_ptr[brow], nb = a.row_ptr[brow + 1] - p0;
    const int n = nb << a.blk_shift;
    const T* xz = reinterpret_cast<const T*>(a.x) + z * a.x_sz;
    T* out = reinterpret_cast<T*>(a.out) + (long)z * a.n_brow * BLK + R;
    float res = 0.f;
    if (n > 0) {
        if (a.op == 1) {
            float s = 0.f;
            for (int e = lane; e < n; e += 64)
                s += Elem<T>::to_f32(xz[(long)a.row_blk[p0 + (e >> a.blk_shift)] * (BLK * BLK) + rl * BLK + (e & (BLK - 1))]);
            res = wave_sum(s);
        } else {
            float mx = -INFINITY;
            for (int e = lane; e < n; e += 64)
                mx = fmaxf(mx, Elem<T>::to_f32(xz[(long)a.row_blk[p0 + (e >> a.blk_shift)] * (BLK * BLK) + rl * BLK + (e & (BLK - 1))]));
            mx = wave_max(mx);
            float s = 0.f;
            for (int e = lane; e < n; e += 64)
                s += expf(Elem<T>::to_f32(xz[(long)a.row_blk[p0 + (e >> a.blk_shift)] * (BLK * BLK) + rl * BLK + (e & (BLK - 1))]) - mx);
            s = wave_sum(s);
            res = (mx == -INFINITY) ? -INFINITY : mx + logf(s);
        }
    }
    if (lane == 0) *out = Elem<T>::from_f32(res);
}

// ---------------------------------------------------------------------------------------
// host side dispatch
// ---------------------------------------------------------------------------------------
static int blk_shift_of(int blk) {
    switch (blk) { case 16: return 4; case 32: return 5; case 64: return 6; case 128: return 7; default: return -1; }
}

#define BS_DISPATCH_BLK(KERN, T, GRID, ARGS)                                               \
    switch (blk) {                                                                         \
        case 16: hipLaunchKernelGGL((KERN<T, 16>), GRID, dim3(256), 0, st, ARGS); break;   \
        case 32: hipLaunchKernelGGL((KERN<T, 32>), GRID, dim3(256), 0, st, ARGS); break;   \
        case 64: hipLaunchKernelGGL((KERN<T, 64>), GRID, dim3(256), 0, st, ARGS); break;   \
        case 128: hipLaunchKernelGGL((KERN<T, 128>), GRID, dim3(256), 0, st, ARGS); break; \
    }
#define BS_DISPATCH(KERN, GRID, ARGS)                                                      \
    switch (dtype) {                                                                       \
        case F32: BS_DISPATCH_BLK(KERN, float, GRID, ARGS) break;                          \
        case BF16: BS_DISPATCH_BLK(KERN, bf16_t, GRID, ARGS) break;                        \
        case F16: BS_DISPATCH_BLK(KERN, f16_t, GRID, ARGS) break;                          \
    }

static long waves_to_blocks(long waves) { return (waves + 3) / 4; }

}  // namespace flyhip

using namespace flyhip;

static int check_common(const char* who, int blk, int dtype, int Z) {
    FLY_REQUIRE(blk_shift_of(blk) >= 0, "%s: block size %d not in {16,32,64,128}", who, blk);
    FLY_REQUIRE(dtype == F32 || dtype == BF16 || dtype == F16, "%s: unknown dtype code %d", who, dtype);
    FLY_REQUIRE(Z >= 1 && Z <= 65535, "%s: batch %d outside [1, 65535]", who, Z);
    return OK;
}

extern "C" int flyhip_bs_sdd(const void* a, const void* b, void* c, const int32_t* lut, int nnz,
                             const int32_t* row_ptr, const int32_t* row_blk, const int32_t* row_col,
                             int n_brow, int brows_per_head,
                             const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                             int Z, int K, int blk,
                             int64_t a_sz, int64_t a_sh, int64_t a_sm, int64_t a_sk,
                             int64_t b_sz, int64_t b_sh, int64_t b_sn, int64_t b_sk,
                             int dtype, void* stream) {
    int rc = check_common("bs_sdd", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(a && b && c && lut, "bs_sdd: null pointer");
    FLY_REQUIRE(nnz >= 0, "bs_sdd: negative nnz");
    FLY_REQUIRE(K > 0 && K % 16 == 0, "bs_sdd: reduction size %d must be a positive multiple of 16", K);
    if (a_sk == 1) FLY_REQUIRE(((a_sz | a_sh | a_sm) % 4) == 0, "bs_sdd: A strides must be multiples of 4 elements");
    if (b_sk == 1) FLY_REQUIRE(((b_sz | b_sh | b_sn) % 4) == 0, "bs_sdd: B strides must be multiples of 4 elements");
    if (nnz == 0) return OK;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    if (row_ptr && row_blk && row_col && blk == 32 && (dtype == BF16 || dtype == F16) && a_sk == 1 && b_sk == 1 &&
        K % 32 == 0 && K <= 128 && ((a_sz | a_sh | a_sm | b_sz | b_sh | b_sn) % 8) == 0 && n_brow > 0 &&
        brows_per_head > 0) {
        FLY_REQUIRE(n_brow % brows_per_head == 0, "bs_sdd: %d block-rows do not divide into heads of %d", n_brow, brows_per_head);
        const int n_heads = n_brow / brows_per_head;
        if (uni_ptr && uni_inner && uni_blk) {
            const int gph = (brows_per_head + 3) / 4;
            SddUniArgs ua{a, b, c, uni_ptr, uni_inner, uni_blk, nnz, brows_per_head, gph, n_heads, Z,
                          a_sz, a_sh, a_sm, b_sz, b_sh, b_sn, nullptr, nullptr, 1.f};
            const long nwg = unit_grid((long)n_heads * Z, gph);
            ua.n_xcd = machine().xcds;
            FLY_REQUIRE(nwg <= 2147483647L, "bs_sdd: too many workgroups");
            dim3 grid((unsigned)nwg);
#define SDD32U_LAUNCH(T)                                                                         \
            switch (K / 32) {                                                                    \
                case 1: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 1>), grid, dim3(256), 0, st, ua); break; \
                case 2: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 2>), grid, dim3(256), 0, st, ua); break; \
                case 3: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 3>), grid, dim3(256), 0, st, ua); break; \
                default: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 4>), grid, dim3(256), 0, st, ua); break; \
            }
            if (dtype == BF16) { SDD32U_LAUNCH(bf16_t) } else { SDD32U_LAUNCH(f16_t) }
#undef SDD32U_LAUNCH
            return check_launch("bs_sdd32u_kernel");
        }
        SddRowArgs ra{a, b, c, row_ptr, row_blk, row_col, nnz, K, brows_per_head, n_heads, Z, a_sz, a_sh, a_sm, b_sz, b_sh, b_sn};
        const long nwg = unit_grid((long)n_heads * Z, (brows_per_head + 3) / 4);
        ra.n_xcd = machine().xcds;
        FLY_REQUIRE(nwg <= 2147483647L, "bs_sdd: too many workgroups");
        dim3 grid((unsigned)nwg);
#define SDD32_LAUNCH(T)                                                                         \
        switch (K / 32) {                                                                       \
            case 1: hipLaunchKernelGGL((bs_sdd32_kernel<T, 1>), grid, dim3(256), 0, st, ra); break; \
            case 2: hipLaunchKernelGGL((bs_sdd32_kernel<T, 2>), grid, dim3(256), 0, st, ra); break; \
            case 3: hipLaunchKernelGGL((bs_sdd32_kernel<T, 3>), grid, dim3(256), 0, st, ra); break; \
            default: hipLaunchKernelGGL((bs_sdd32_kernel<T, 4>), grid, dim3(256), 0, st, ra); break; \
        }
        if (dtype == BF16) { SDD32_LAUNCH(bf16_t) } else { SDD32_LAUNCH(f16_t) }
#undef SDD32_LAUNCH
        return check_launch("bs_sdd32_kernel");
    }
    SddArgs args{a, b, c, lut, nnz, K, a_sz, a_sh, a_sm, a_sk, b_sz, b_sh, b_sn, b_sk};
    const int tile = blk >= 32 ? 32 : 16, sub = blk / tile;
    const long nblocks = waves_to_blocks((long)nnz * sub * sub);
    FLY_REQUIRE(nblocks <= 2147483647L, "bs_sdd: too many blocks");
    dim3 grid((unsigned)nblocks, Z);
    BS_DISPATCH(bs_sdd_kernel, grid, args)
    return check_launch("bs_sdd_kernel");
}

template <int EPI>
static int launch_sdd_epilogue(const char* what, const void* a_dn, const void* b_dn, const void* p, const float* rowvec, void* c,
                               const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                               int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                               int64_t a_sz, int64_t a_sh, int64_t a_sm, int64_t b_sz, int64_t b_sh, int64_t b_sn,
                               float scale, int dtype, void* stream, const SddUniArgs* second = nullptr) {
    int rc = check_common(what, blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(a_dn && b_dn && (EPI != 1 || p) && (rowvec || (EPI == 3 && second && second->out)) && c && uni_ptr &&
                uni_inner && uni_blk, "%s: null pointer", what);
    FLY_REQUIRE(blk == 32 && (dtype == BF16 || dtype == F16), "%s: needs 32x32 blocks of bf16 / fp16", what);
    FLY_REQUIRE(K % 32 == 0 && K >= 32 && K <= 128, "%s: head dim %d not a multiple of 32 up to 128", what, K);
    FLY_REQUIRE(nnz > 0 && n_heads > 0 && brows_per_head > 0, "%s: bad sizes", what);
    FLY_REQUIRE(((a_sz | a_sh | a_sm | b_sz | b_sh | b_sn) % 8) == 0, "%s: strides must be multiples of 8 elements", what);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    const int gph = (brows_per_head + 3) / 4;
    SddUniArgs ua{a_dn, b_dn, c, uni_ptr, uni_inner, uni_blk, nnz, brows_per_head, gph, n_heads, Z,
                  a_sz, a_sh, a_sm, b_sz, b_sh, b_sn, p, rowvec, scale};
    if (EPI == 3) {
        FLY_REQUIRE(second && second->a2 && second->b2 && second->lse2 && second->p2, "%s: null pointer", what);
        FLY_REQUIRE(((second->a2_sz | second->a2_sh | second->a2_sm | second->b2_sz | second->b2_sh | second->b2_sn) % 8) == 0,
                    "%s: strides must be multiples of 8 elements", what);
        ua.a2 = second->a2; ua.b2 = second->b2; ua.lse2 = second->lse2; ua.p2 = second->p2; ua.scale2 = second->scale2;
        ua.a2_sz = second->a2_sz; ua.a2_sh = second->a2_sh; ua.a2_sm = second->a2_sm;
        ua.b2_sz = second->b2_sz; ua.b2_sh = second->b2_sh; ua.b2_sn = second->b2_sn;
        FLY_REQUIRE(second->dq && ((second->dq_sz | second->dq_sh | second->dq_sm) % 4) == 0,
                    "%s: dq missing or its strides are not multiples of 4 elements", what);
        ua.dq = second->dq; ua.dq_sz = second->dq_sz; ua.dq_sh = second->dq_sh; ua.dq_sm = second->dq_sm;
        FLY_REQUIRE(!second->out || ((second->o_sz | second->o_sh | second->o_sm) % 8) == 0,
                    "%s: out strides must be multiples of 8 elements", what);
        ua.out = second->out; ua.o_sz = second->o_sz; ua.o_sh = second->o_sh; ua.o_sm = second->o_sm;
    }
    const long nwg = unit_grid((long)n_heads * Z, gph);
    ua.n_xcd = machine().xcds;
    FLY_REQUIRE(nwg <= 2147483647L, "%s: too many workgroups", what);
    dim3 grid((unsigned)nwg);
#define SDDS_LAUNCH(T)                                                                                  \
    switch (K / 32) {                                                                                   \
        case 1: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 1, EPI>), grid, dim3(256), 0, st, ua); break;  \
        case 2: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 2, EPI>), grid, dim3(256), 0, st, ua); break;  \
        case 3: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 3, EPI>), grid, dim3(256), 0, st, ua); break;  \
        default: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 4, EPI>), grid, dim3(256), 0, st, ua); break; \
    }
    if constexpr (EPI == 3) {
        if (second->drop_thresh != 0u) {
            ua.drop_seed = second->drop_seed; ua.drop_thresh = second->drop_thresh; ua.drop_scale = second->drop_scale;
            FLY_REQUIRE((long)Z * n_heads * brows_per_head * 32 <= 4294967295L, "%s: more than 2^32 rows", what);
#define SDDS_DROP_LAUNCH(T)                                                                                   \
    switch (K / 32) {                                                                                         \
        case 1: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 1, 3, true>), grid, dim3(256), 0, st, ua); break;    \
        case 2: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 2, 3, true>), grid, dim3(256), 0, st, ua); break;    \
        case 3: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 3, 3, true>), grid, dim3(256), 0, st, ua); break;    \
        default: hipLaunchKernelGGL((bs_sdd32u_kernel<T, 4, 3, true>), grid, dim3(256), 0, st, ua); break;   \
    }
            if (dtype == BF16) { SDDS_DROP_LAUNCH(bf16_t) } else { SDDS_DROP_LAUNCH(f16_t) }
#undef SDDS_DROP_LAUNCH
            return check_launch(what);
        }
    }
    if (dtype == BF16) { SDDS_LAUNCH(bf16_t) } else { SDDS_LAUNCH(f16_t) }
#undef SDDS_LAUNCH
    return check_launch(what);
}

extern "C" int flyhip_bs_sdd_dsoftmax(const void* dout, const void* v, const void* p, const float* delta, void* ds,
                                      const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                                      int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                                      int64_t a_sz, int64_t a_sh, int64_t a_sm,
                                      int64_t b_sz, int64_t b_sh, int64_t b_sn,
                                      float scale, int dtype, void* stream) {
    return launch_sdd_epilogue<1>("bs_sdd_dsoftmax", dout, v, p, delta, ds, uni_ptr, uni_inner, uni_blk, nnz, n_heads,
                                  brows_per_head, Z, K, blk, a_sz, a_sh, a_sm, b_sz, b_sh, b_sn, scale, dtype, stream);
}

extern "C" int flyhip_bs_sdd_prob_dsoftmax_dropout(const void* dout, const void* v, const void* q, const void* k,
                                           const float* delta, const void* out, const float* lse2, void* ds, void* p, void* dq,
                                           const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                                           int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                                           int64_t do_sz, int64_t do_sh, int64_t do_sm,
                                           int64_t v_sz, int64_t v_sh, int64_t v_sn,
                                           int64_t q_sz, int64_t q_sh, int64_t q_sm,
                                           int64_t k_sz, int64_t k_sh, int64_t k_sn,
                                           int64_t dq_sz, int64_t dq_sh, int64_t dq_sm,
                                           int64_t o_sz, int64_t o_sh, int64_t o_sm,
                                           float scale, int dtype, float dropout_p, uint64_t dropout_seed, void* stream);

extern "C" int flyhip_bs_sdd_prob_dsoftmax(const void* dout, const void* v, const void* q, const void* k,
                                           const float* delta, const void* out, const float* lse2, void* ds, void* p, void* dq,
                                           const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                                           int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                                           int64_t do_sz, int64_t do_sh, int64_t do_sm,
                                           int64_t v_sz, int64_t v_sh, int64_t v_sn,
                                           int64_t q_sz, int64_t q_sh, int64_t q_sm,
                                           int64_t k_sz, int64_t k_sh, int64_t k_sn,
                                           int64_t dq_sz, int64_t dq_sh, int64_t dq_sm,
                                           int64_t o_sz, int64_t o_sh, int64_t o_sm,
                                           float scale, int dtype, void* stream) {
    return flyhip_bs_sdd_prob_dsoftmax_dropout(dout, v, q, k, delta, out, lse2, ds, p, dq, uni_ptr, uni_inner, uni_blk, nnz,
                                               n_heads, brows_per_head, Z, K, blk, do_sz, do_sh, do_sm, v_sz, v_sh, v_sn,
                                               q_sz, q_sh, q_sm, k_sz, k_sh, k_sn, dq_sz, dq_sh, dq_sm, o_sz, o_sh, o_sm,
                                               scale, dtype, 0.f, 0, stream);
}

extern "C" int flyhip_bs_sdd_prob_dsoftmax_dropout(const void* dout, const void* v, const void* q, const void* k,
                                           const float* delta, const void* out, const float* lse2, void* ds, void* p, void* dq,
                                           const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                                           int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                                           int64_t do_sz, int64_t do_sh, int64_t do_sm,
                                           int64_t v_sz, int64_t v_sh, int64_t v_sn,
                                           int64_t q_sz, int64_t q_sh, int64_t q_sm,
                                           int64_t k_sz, int64_t k_sh, int64_t k_sn,
                                           int64_t dq_sz, int64_t dq_sh, int64_t dq_sm,
                                           int64_t o_sz, int64_t o_sh, int64_t o_sm,
                                           float scale, int dtype, float dropout_p, uint64_t dropout_seed, void* stream) {
    FLY_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "bs_sdd_prob_dsoftmax: dropout_p %g not in [0, 1)", (double)dropout_p);
    SddUniArgs second{};
    const DropArgs drop = drop_args(dropout_p, dropout_seed);
    second.drop_seed = drop.seed; second.drop_thresh = drop.thresh; second.drop_scale = drop.scale;
    second.out = out; second.o_sz = o_sz; second.o_sh = o_sh; second.o_sm = o_sm;
    second.dq = dq; second.dq_sz = dq_sz; second.dq_sh = dq_sh; second.dq_sm = dq_sm;
    second.a2 = q; second.b2 = k; second.lse2 = lse2; second.p2 = p; second.scale2 = scale * 1.4426950408889634f;
    second.a2_sz = q_sz; second.a2_sh = q_sh; second.a2_sm = q_sm;
    second.b2_sz = k_sz; second.b2_sh = k_sh; second.b2_sn = k_sn;
    return launch_sdd_epilogue<3>("bs_sdd_prob_dsoftmax", dout, v, nullptr, delta, ds, uni_ptr, uni_inner, uni_blk, nnz,
                                  n_heads, brows_per_head, Z, K, blk, do_sz, do_sh, do_sm, v_sz, v_sh, v_sn, scale, dtype,
                                  stream, &second);
}

// ---------------------------------------------------------------------------------------
// gradients of the one-kernel block-sparse attention without the probabilities in memory
// ---------------------------------------------------------------------------------------
// With P = 2^(scale log2e q.k - lse2[query]) on the nonzero 32 x 32 blocks, g = d out and delta = rowsum(g * out):
// d v = P^T g, dS = P (g v^T - delta), d q = scale dS k, d k = scale dS^T q.  One kernel in two orientations, neither
// of which writes P or dS: a workgroup owns four block-rows (query-major: d q, and delta on the way) or four
// block-columns (key-major: d k and d v), a wave one of them with its two operands in registers (q and g rows; k and v
// rows), and walks the union of their lists (union_table, transposed for key-major), every 32-row tile of the other
// side (K with V; Q with g, lse2 and delta) moved once straight into LDS for the four waves.  Per block S^T = Y1 . x1 and
// delta - G^T = delta - Y2 . x2 (x2 negated, the sums start at delta; a lane's results over the two 16-row blocks are inner rows
// 4 g + i and 16 + 4 g + i, the contraction slots of what follows), then d x^T[e][outer] += Y^T[e][inner] . {-dS, P}[inner][outer]
// with Y^T fragments by transposing LDS reads of the same tiles.
struct AttnBwdArgs {
    const void* q; const void* k; const void* v; const void* go; const void* out;
    const float* lse2; float* delta;                 // (Z, H, 32 * query blocks); delta is written by the query-major launch
    void* dq; void* dk; void* dv;
    const int32_t* uni_ptr; const int32_t* uni_inner; const int32_t* uni_blk;      // of the launch's orientation
    int outer_blocks, inner_blocks, q_blocks, grps_per_head, n_heads, Z;
    long q_sz, q_sh, q_sm, k_sz, k_sh, k_sm, v_sz, v_sh, v_sm, g_sz, g_sh, g_sm, o_sz, o_sh, o_sm;
    long dq_sz, dq_sh, dq_sm, dk_sz, dk_sh, dk_sm, dv_sz, dv_sh, dv_sm;
    float scale;
    int n_xcd;
    // DROP: the forward dropped probabilities by the hash of (seed, row = (z H + head) L + query, key) (drop_keep): d v takes
    // m P and dS = P (m g.v - delta), m = 0 or 1 / (1 - p)
    uint32_t drop_seed, drop_thresh; float drop_scale;
    // the forward's additive masks (flyhip_bs_attn_masks), optional: key_mask (Z, keys) and attn_mask (queries, keys),
    // float32, added to scale * q.k (0 / -inf, or any finite bias)
    const float* key_mask; long km_stride; const float* attn_mask; long am_stride;
};

// Bound by the vector ALU (70 % of the cycles query-major with dropout, 60 % key-major) and the matrix pipe (26 - 43 %) taking turns at
// two to three waves per SIMD; LDS 15 - 27 %, without bank conflicts since the tiles go straight into LDS with swizzled rows.
// B=8, 12 heads of 4096 tokens, 64 dims, training step in bfloat16: 797 -> 727 us, with dropout 1077 -> 1003 (tiles by way of
// registers into padded rows, list entries by vector loads, a product per pair for the dropout scale before).
// (registers for three waves per SIMD: the key-major form at 64 dims takes more without the bound, two waves per SIMD; with the
//  dropout hashes it would spill inside the loop at that bound and keeps two.  Measured and not kept: tiles asked for two steps
//  ahead, 2 % slower; one outer block after the other with fragment reads of its own, which leaves room for a fourth wave
//  query-major, 5 % slower, as are four waves with spills)
// MASKED: a variant of its own, so that the kernels without masks carry nothing of them (as a kernel-uniform branch the
// mask code cost the key-major form 35 more spilled registers and the query-major form a wave per SIMD)
template <typename T, int E, bool KEYMAJOR, bool DROP = false, bool MASKED = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KEYMAJOR && (DROP || MASKED) ? 2 : 3, 8))) void bs_attn32_bwd_kernel(const AttnBwdArgs a) {
    static_assert(!(DROP && MASKED), "the forward with masks has no dropout");
    static_assert(sizeof(T) == 2 && E % 32 == 0, "2-byte inputs, whole MFMA steps");
    constexpr int KS = E / 32, EB = E / 16, ROWB = 2 * E, TILE = 32 * ROWB;
    constexpr float LOG2E = 1.4426950408889634f;
    __shared__ __attribute__((aligned(128))) char tiles[2][2][TILE];            // [stage][Y1 | Y2], rows as RowsToLds leaves them
    __shared__ __attribute__((aligned(16))) float rowv[2][3][32];              // key-major: [stage][lse2 (DROP: - log2 drop_scale) | delta (DROP: / drop_scale) | row hash] of the tile's queries
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int unit, grp;
    if (!unit_of(blockIdx.x, a.n_xcd, a.grps_per_head, a.n_heads * a.Z, unit, grp)) return;
    const int z = unit / a.n_heads, head = unit % a.n_heads;
    const int ug = head * a.grps_per_head + grp;
    const int p0 = a.uni_ptr[ug], n = a.uni_ptr[ug + 1] - p0;
    const int bo = grp * 4 + w;
    const bool have = bo < a.outer_blocks;
    const int bo_c = min(bo, a.outer_blocks - 1);
    const uint16_t* qz = reinterpret_cast<const uint16_t*>(a.q) + z * a.q_sz + head * a.q_sh;
    const uint16_t* kz = reinterpret_cast<const uint16_t*>(a.k) + z * a.k_sz + head * a.k_sh;
    const uint16_t* vz = reinterpret_cast<const uint16_t*>(a.v) + z * a.v_sz + head * a.v_sh;
    const uint16_t* gz = reinterpret_cast<const uint16_t*>(a.go) + z * a.g_sz + head * a.g_sh;
    const uint16_t* x1p = KEYMAJOR ? kz : qz;  const long x1s = KEYMAJOR ? a.k_sm : a.q_sm;     // outer operands
    const uint16_t* x2p = KEYMAJOR ? vz : gz;  const long x2s = KEYMAJOR ? a.v_sm : a.g_sm;
    const uint16_t* y1p = KEYMAJOR ? qz : kz;  const long y1s = KEYMAJOR ? a.q_sm : a.k_sm;     // inner tiles
    const uint16_t* y2p = KEYMAJOR ? gz : vz;  const long y2s = KEYMAJOR ? a.g_sm : a.v_sm;
    const long qvec = ((long)z * a.n_heads + head) * a.q_blocks * 32;                          // row vectors of this (z, head)
    T* d1 = KEYMAJOR ? reinterpret_cast<T*>(a.dk) + z * a.dk_sz + head * a.dk_sh : reinterpret_cast<T*>(a.dq) + z * a.dq_sz + head * a.dq_sh;
    const long d1s = KEYMAJOR ? a.dk_sm : a.dq_sm;
    T* d2 = reinterpret_cast<T*>(a.dv) + z * a.dv_sz + head * a.dv_sh;

    // dS = P (M g.v - delta), M = drop_scale or 0, is formed as -P' (delta / drop_scale - kept g.v) with P' = drop_scale P: the sums
    // start at delta / drop_scale, x2 goes in negated and the factor of P' is in the rows' exponents, so that a pair costs one
    // select and one product.  (The second products read M P and dS themselves rounded to the input type: float16 without the factor
    // would put them log2(drop_scale) bits deeper into its subnormal range.)
    const float inv_drop = DROP ? 1.0f / a.drop_scale : 1.0f, log_drop = DROP ? log2f(a.drop_scale) : 0.f;
    uintx4 x1[2][KS], x2[2][KS];
    float l_own[2] = {0.f, 0.f}, d_own[2] = {0.f, 0.f};          // query-major: lse2 and delta of the lane's queries, as in rowv
    float km_own[2] = {0.f, 0.f};                     // key-major: the key mask entries of the lane's keys
    uint32_t h_own[2] = {0u, 0u};                     // DROP, query-major: hash of (seed, global row) of the lane's queries
    floatx4 acc1[2][EB], acc2[KEYMAJOR ? 2 : 1][KEYMAJOR ? EB : 1];     // d q | d k, and d v
#pragma unroll
    for (int qq = 0; qq < 2; ++qq) {
        const long row = (long)bo_c * 32 + 16 * qq + r16;
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            x1[qq][c] = *reinterpret_cast<const uintx4*>(x1p + row * x1s + 32 * c + 8 * g);
            x2[qq][c] = *reinterpret_cast<const uintx4*>(x2p + row * x2s + 32 * c + 8 * g);
        }
        if (MASKED && KEYMAJOR && a.key_mask) km_own[qq] = a.key_mask[z * a.km_stride + row];
        if (!KEYMAJOR) {
            l_own[qq] = a.lse2[qvec + row] - log_drop;
            if (DROP) h_own[qq] = drop_row_hash(a.drop_seed, (uint32_t)(qvec + row));
            // delta of the query, g . out, from the output row in the layout of the gradient row; kept for the key-major launch
            const uint16_t* orow = reinterpret_cast<const uint16_t*>(a.out) + z * a.o_sz + head * a.o_sh + row * a.o_sm;
            float part = 0.f;
#pragma unroll
            for (int c = 0; c < KS; ++c) {
                const uintx4 ov = *reinterpret_cast<const uintx4*>(orow + 32 * c + 8 * g);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    T x, y;
                    *reinterpret_cast<uint16_t*>(&x) = (uint16_t)(x2[qq][c][e >> 1] >> (16 * (e & 1)));
                    *reinterpret_cast<uint16_t*>(&y) = (uint16_t)(ov[e >> 1] >> (16 * (e & 1)));
                    part += Elem<T>::to_f32(x) * Elem<T>::to_f32(y);
                }
            }
            part = group_sum(part);
            d_own[qq] = DROP ? part * inv_drop : part;
            if (have && g == 0) a.delta[qvec + row] = part;
        }
#pragma unroll
        for (int c = 0; c < KS; ++c) x2[qq][c] ^= 0x80008000u;
#pragma unroll
        for (int eb = 0; eb < EB; ++eb) acc1[qq][eb] = Frag<float>::zero();
    }
    if (KEYMAJOR) {
#pragma unroll
        for (int qq = 0; qq < 2; ++qq)
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) acc2[qq][eb] = Frag<float>::zero();
    }

    RowsToLds<32, E, 256> r1, r2;
    r1.init(y1p, y1s, 32 * a.inner_blocks - 1, w, lane);
    r2.init(y2p, y2s, 32 * a.inner_blocks - 1, w, lane);
    float rl = 0.f, rd = 0.f;
    uint32_t rh = 0u;
    auto fetch = [&](int inner, int stage) __attribute__((always_inline)) {
        r1.fetch(32 * inner, tiles[stage][0], w, lane);
        r2.fetch(32 * inner, tiles[stage][1], w, lane);
        if (KEYMAJOR && tid < 32) {
            const long at = qvec + (long)inner * 32 + tid;
            rl = a.lse2[at];
            rd = a.delta[at];
            if (DROP) rh = drop_row_hash(a.drop_seed, (uint32_t)at);
        }
    };
    auto stash = [&](int stage) __attribute__((always_inline)) {
        if (KEYMAJOR && tid < 32) {
            rowv[stage][0][tid] = rl - log_drop;
            rowv[stage][1][tid] = DROP ? rd * inv_drop : rd;
            if (DROP) rowv[stage][2][tid] = __uint_as_float(rh);
        }
    };
    const float sc = a.scale * LOG2E;
    // row fragments: chunk 4 c + g of row 16 hb + r16; transposing reads: rows 4 g + r16 / 4 (+ 16), half r16 % 2 of chunk
    // 2 eb + (r16 % 4) / 2 (the swizzle depends on the row modulo 16 alone)
    const int trow = 4 * g + (r16 >> 2);
    int foff[KS], toff[EB];
#pragma unroll
    for (int c = 0; c < KS; ++c) foff[c] = r16 * ROWB + rows_swz(r16, 4 * c + g, ROWB) * 16;
#pragma unroll
    for (int eb = 0; eb < EB; ++eb) toff[eb] = trow * ROWB + rows_swz(trow, 2 * eb + ((r16 & 3) >> 1), ROWB) * 16 + 8 * (r16 & 1);
    // (list entries a step ahead of their use)
    int inner_cur = n > 0 ? table_entry(a.uni_inner + p0) : 0, inner_next = n > 1 ? table_entry(a.uni_inner + p0 + 1) : 0;
    int blk_cur = n > 0 ? table_entry(a.uni_blk + (long)p0 * 4 + w) : -1;
    if (n > 0) {
        fetch(inner_cur, 0);
        stash(0);
    }
    drain_loads();
    __syncthreads();
    for (int s = 0; s < n; ++s) {
        const int cur = s & 1;
        const bool more = s + 1 < n;
        if (more) fetch(inner_next, cur ^ 1);
        const int blk_next = table_entry(a.uni_blk + (long)(p0 + min(s + 1, n - 1)) * 4 + w);
        const int inner_after = table_entry(a.uni_inner + p0 + min(s + 2, n - 1));
        const bool present = have && blk_cur >= 0;               // wave-uniform
        if (present) {
            const char* Y1 = tiles[cur][0];
            const char* Y2 = tiles[cur][1];
            floatx4 s1[2][2], gp[2][2], nd[2];           // [outer block][inner block hb]: scores (unscaled) and delta - g.v
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                if (KEYMAJOR) nd[hb] = *reinterpret_cast<const floatx4*>(&rowv[cur][1][16 * hb + 4 * g]);
#pragma unroll
                for (int qq = 0; qq < 2; ++qq) {
                    s1[qq][hb] = Frag<float>::zero();
                    gp[qq][hb] = KEYMAJOR ? nd[hb] : floatx4{d_own[qq], d_own[qq], d_own[qq], d_own[qq]};
                }
            }
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int c = 0; c < KS; ++c) {
                    const int off = 16 * hb * ROWB + foff[c];
                    const uintx4 f1 = *reinterpret_cast<const uintx4*>(Y1 + off);
                    const uintx4 f2 = *reinterpret_cast<const uintx4*>(Y2 + off);
#pragma unroll
                    for (int qq = 0; qq < 2; ++qq) {
                        s1[qq][hb] = mma32<T>(f1, x1[qq][c], s1[qq][hb]);
                        gp[qq][hb] = mma32<T>(f2, x2[qq][c], gp[qq][hb]);
                    }
                }
            floatx4 ln4[2], hh4[2];                      // key-major: the tile's queries' lse2 and row hashes, by block
            if (KEYMAJOR) {
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    ln4[hb] = *reinterpret_cast<const floatx4*>(&rowv[cur][0][16 * hb + 4 * g]);
                    if (DROP) hh4[hb] = *reinterpret_cast<const floatx4*>(&rowv[cur][2][16 * hb + 4 * g]);
                }
            }
            if constexpr (MASKED) {                                     // the masks, in units of the unscaled scores
                const float inv_scale = 1.0f / a.scale;
#pragma unroll
                for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb) {
                        const long in0 = (long)inner_cur * 32 + 16 * hb + 4 * g;        // the element's four inner rows
                        const long orow = (long)bo_c * 32 + 16 * qq + r16;             // its outer row
                        floatx4 add = Frag<float>::zero();
                        if (!KEYMAJOR) {
                            if (a.key_mask) add += *reinterpret_cast<const floatx4*>(a.key_mask + z * a.km_stride + in0);
                            if (a.attn_mask) add += *reinterpret_cast<const floatx4*>(a.attn_mask + orow * a.am_stride + in0);
                        } else {
                            if (a.key_mask) add += km_own[qq];
                            if (a.attn_mask) {
#pragma unroll
                                for (int i = 0; i < 4; ++i) add[i] += a.attn_mask[(in0 + i) * a.am_stride + orow];
                            }
                        }
                        s1[qq][hb] += add * inv_scale;
                    }
            }
#pragma unroll
            for (int qq = 0; qq < 2; ++qq)
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    uint32_t r01 = 0u, r23 = 0u;         // key-major: 16 bits a query, see drop_halves_of_column
                    if (KEYMAJOR && DROP)
                        drop_halves_of_column(__float_as_uint((r16 & 1) ? hh4[hb][2] : hh4[hb][0]), __float_as_uint((r16 & 1) ? hh4[hb][3] : hh4[hb][1]),
                                              (uint32_t)bo_c * 32u + 16u * qq + r16, r01, r23);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float lrow = KEYMAJOR ? ln4[hb][i] : l_own[qq];
                        const float pr = __builtin_amdgcn_exp2f(fmaf(s1[qq][hb][i], sc, -lrow));   // (a row without scores: lse2 = +inf)
                        if (DROP) {
                            // (query, key) of the element: the inner row 16 hb + 4 g + i of the tile, the outer row 16 qq + r16
                            bool keep;
                            if (KEYMAJOR) {
                                const uint32_t pair = i < 2 ? r01 : r23;
                                keep = ((i & 1) ? pair >> 16 : pair & 0xffffu) >= a.drop_thresh;
                            } else {
                                keep = drop_keep(h_own[qq], (uint32_t)inner_cur * 32u + 16u * hb + 4u * g + i, a.drop_thresh);
                            }
                            s1[qq][hb][i] = keep ? pr : 0.f;
                            gp[qq][hb][i] = pr * (keep ? gp[qq][hb][i] : KEYMAJOR ? nd[hb][i] : d_own[qq]);
                        } else {
                            s1[qq][hb][i] = pr;
                            gp[qq][hb][i] *= pr;
                        }
                    }
                }
            uintx4 pb[KEYMAJOR ? 2 : 1], sb[2];
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) {
                sb[qq] = uintx4{pack2<T>(gp[qq][0][0], gp[qq][0][1]), pack2<T>(gp[qq][0][2], gp[qq][0][3]),
                                pack2<T>(gp[qq][1][0], gp[qq][1][1]), pack2<T>(gp[qq][1][2], gp[qq][1][3])};
                if (KEYMAJOR)
                    pb[qq] = uintx4{pack2<T>(s1[qq][0][0], s1[qq][0][1]), pack2<T>(s1[qq][0][2], s1[qq][0][3]),
                                    pack2<T>(s1[qq][1][0], s1[qq][1][1]), pack2<T>(s1[qq][1][2], s1[qq][1][3])};
            }
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) {
                const uintx4 t1 = lds_read_tr8(Y1 + toff[eb], Y1 + toff[eb] + 16 * ROWB);
#pragma unroll
                for (int qq = 0; qq < 2; ++qq) acc1[qq][eb] = mma32<T>(t1, sb[qq], acc1[qq][eb]);
                if (KEYMAJOR) {
                    const uintx4 t2 = lds_read_tr8(Y2 + toff[eb], Y2 + toff[eb] + 16 * ROWB);
#pragma unroll
                    for (int qq = 0; qq < 2; ++qq) acc2[qq][eb] = mma32<T>(t2, pb[qq], acc2[qq][eb]);
                }
            }
        }
        if (more) stash(cur ^ 1);
        inner_cur = inner_next;
        inner_next = inner_after;
        blk_cur = blk_next;
        drain_loads();                                   // this wave's share of the next tile is in LDS
        __syncthreads();
    }
    if (have) {
#pragma unroll
        for (int qq = 0; qq < 2; ++qq) {
            const long row = (long)bo * 32 + 16 * qq + r16;
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) store4_f32(d1 + row * d1s + 16 * eb + 4 * g, acc1[qq][eb] * -a.scale);
            if (KEYMAJOR) {
#pragma unroll
                for (int eb = 0; eb < EB; ++eb) store4_f32(d2 + row * a.dv_sm + 16 * eb + 4 * g, acc2[qq][eb]);
            }
        }
    }
}

template <typename T, int E, bool KEYMAJOR, bool DROP, bool MASKED = false>
static int launch_attn_bwd_as(const AttnBwdArgs& a, hipStream_t st) {
    AttnBwdArgs args = a;
    args.n_xcd = machine().xcds;
    const long grid = unit_grid((long)a.n_heads * a.Z, a.grps_per_head);
    if (grid > 2147483647L) return fail(ERR_ARG, "bs_attn_bwd: too many workgroups");
    hipLaunchKernelGGL((bs_attn32_bwd_kernel<T, E, KEYMAJOR, DROP, MASKED>), dim3((unsigned)grid), dim3(256), 0, st, args);
    return check_launch("bs_attn32_bwd_kernel");
}
template <typename T, int E, bool KEYMAJOR>
static int launch_attn_bwd(const AttnBwdArgs& a, hipStream_t st) {
    if (a.key_mask != nullptr || a.attn_mask != nullptr) return launch_attn_bwd_as<T, E, KEYMAJOR, false, true>(a, st);
    return a.drop_thresh != 0u ? launch_attn_bwd_as<T, E, KEYMAJOR, true>(a, st) : launch_attn_bwd_as<T, E, KEYMAJOR, false>(a, st);
}

extern "C" int flyhip_bs_attn_bwd(const void* q, const void* k, const void* v, const void* out, const void* grad_out,
                                  const float* lse2, float* delta, void* dq, void* dk, void* dv,
                                  const int32_t* row_ptr, const int32_t* row_inner, const int32_t* row_blk,
                                  const int32_t* col_ptr, const int32_t* col_inner, const int32_t* col_blk,
                                  int n_heads, int brows_per_head, int bcols_per_head, int Z, int E,
                                  int64_t q_sz, int64_t q_sh, int64_t q_sm, int64_t k_sz, int64_t k_sh, int64_t k_sm,
                                  int64_t v_sz, int64_t v_sh, int64_t v_sm, int64_t o_sz, int64_t o_sh, int64_t o_sm,
                                  int64_t g_sz, int64_t g_sh, int64_t g_sm,
                                  int64_t dq_sz, int64_t dq_sh, int64_t dq_sm, int64_t dk_sz, int64_t dk_sh, int64_t dk_sm,
                                  int64_t dv_sz, int64_t dv_sh, int64_t dv_sm,
                                  float scale, int dtype, float dropout_p, uint64_t dropout_seed,
                                  const float* key_mask, int64_t key_mask_stride, const float* attn_mask, int64_t attn_mask_stride,
                                  void* stream) {
    FLY_REQUIRE(q && k && v && out && grad_out && lse2 && delta && dq && dk && dv, "bs_attn_bwd: null pointer");
    FLY_REQUIRE(scale > 0.f, "bs_attn_bwd: scale must be positive");
    FLY_REQUIRE((!key_mask || key_mask_stride % 4 == 0) && (!attn_mask || attn_mask_stride % 4 == 0) &&
                ((reinterpret_cast<uintptr_t>(key_mask) | reinterpret_cast<uintptr_t>(attn_mask)) % 16) == 0,
                "bs_attn_bwd: mask rows must be 16-byte aligned (strides in multiples of 4 floats)");
    FLY_REQUIRE(dropout_p == 0.f || (!key_mask && !attn_mask), "bs_attn_bwd: no dropout together with masks (the forward has none)");
    FLY_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "bs_attn_bwd: dropout_p %g not in [0, 1)", (double)dropout_p);
    FLY_REQUIRE((long)Z * n_heads * brows_per_head * 32 <= 4294967295L, "bs_attn_bwd: more than 2^32 query rows");
    FLY_REQUIRE(row_ptr && row_inner && row_blk && col_ptr && col_inner && col_blk, "bs_attn_bwd: null table");
    FLY_REQUIRE(n_heads > 0 && brows_per_head > 0 && bcols_per_head > 0 && Z > 0, "bs_attn_bwd: empty problem");
    FLY_REQUIRE(E == 32 || E == 64, "bs_attn_bwd: head dim %d not in {32, 64}", E);
    FLY_REQUIRE(dtype == BF16 || dtype == F16, "bs_attn_bwd supports bfloat16 and float16, got dtype code %d", dtype);
    FLY_REQUIRE(((q_sz | q_sh | q_sm | k_sz | k_sh | k_sm | v_sz | v_sh | v_sm | o_sz | o_sh | o_sm | g_sz | g_sh | g_sm) % 8) == 0,
                "bs_attn_bwd: input strides must be multiples of 8 elements (16-byte loads)");
    FLY_REQUIRE(((dq_sz | dq_sh | dq_sm | dk_sz | dk_sh | dk_sm | dv_sz | dv_sh | dv_sm) % 4) == 0,
                "bs_attn_bwd: output strides must be multiples of 4 elements (8-byte stores)");
    FLY_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
                  reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(grad_out)) % 16) == 0 &&
                ((reinterpret_cast<uintptr_t>(dq) | reinterpret_cast<uintptr_t>(dk) | reinterpret_cast<uintptr_t>(dv)) % 8) == 0,
                "bs_attn_bwd: pointers must be 16-byte (inputs) and 8-byte (outputs) aligned");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    AttnBwdArgs a{};
    a.q = q; a.k = k; a.v = v; a.go = grad_out; a.out = out; a.lse2 = lse2; a.delta = delta; a.dq = dq; a.dk = dk; a.dv = dv;
    a.q_blocks = brows_per_head; a.n_heads = n_heads; a.Z = Z; a.scale = scale;
    const DropArgs drop = drop_args(dropout_p, dropout_seed);
    a.drop_seed = drop.seed; a.drop_thresh = drop.thresh; a.drop_scale = drop.scale;
    a.key_mask = key_mask; a.km_stride = key_mask_stride; a.attn_mask = attn_mask; a.am_stride = attn_mask_stride;
    a.q_sz = q_sz; a.q_sh = q_sh; a.q_sm = q_sm; a.k_sz = k_sz; a.k_sh = k_sh; a.k_sm = k_sm; a.v_sz = v_sz; a.v_sh = v_sh; a.v_sm = v_sm;
    a.g_sz = g_sz; a.g_sh = g_sh; a.g_sm = g_sm; a.o_sz = o_sz; a.o_sh = o_sh; a.o_sm = o_sm;
    a.dq_sz = dq_sz; a.dq_sh = dq_sh; a.dq_sm = dq_sm; a.dk_sz = dk_sz; a.dk_sh = dk_sh; a.dk_sm = dk_sm;
    a.dv_sz = dv_sz; a.dv_sh = dv_sh; a.dv_sm = dv_sm;
    for (int km = 0; km < 2; ++km) {                 // query-major first: it leaves delta for the key-major launch
        a.uni_ptr = km ? col_ptr : row_ptr; a.uni_inner = km ? col_inner : row_inner; a.uni_blk = km ? col_blk : row_blk;
        a.outer_blocks = km ? bcols_per_head : brows_per_head;
        a.inner_blocks = km ? brows_per_head : bcols_per_head;
        a.grps_per_head = (a.outer_blocks + 3) / 4;
        int rc;
#define ATTN_BWD_LAUNCH(TT, EE) rc = km ? launch_attn_bwd<TT, EE, true>(a, st) : launch_attn_bwd<TT, EE, false>(a, st)
        if (dtype == BF16) { if (E == 32) ATTN_BWD_LAUNCH(bf16_t, 32); else ATTN_BWD_LAUNCH(bf16_t, 64); }
        else { if (E == 32) ATTN_BWD_LAUNCH(f16_t, 32); else ATTN_BWD_LAUNCH(f16_t, 64); }
#undef ATTN_BWD_LAUNCH
        if (rc) return rc;
    }
    return 0;
}

extern "C" int flyhip_bs_sdd_prob(const void* q, const void* k, const float* lse2, void* p,
                                  const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                                  int nnz, int n_heads, int brows_per_head, int Z, int K, int blk,
                                  int64_t a_sz, int64_t a_sh, int64_t a_sm,
                                  int64_t b_sz, int64_t b_sh, int64_t b_sn,
                                  float scale, int dtype, void* stream) {
    return launch_sdd_epilogue<2>("bs_sdd_prob", q, k, nullptr, lse2, p, uni_ptr, uni_inner, uni_blk, nnz, n_heads,
                                  brows_per_head, Z, K, blk, a_sz, a_sh, a_sm, b_sz, b_sh, b_sn,
                                  scale * 1.4426950408889634f, dtype, stream);
}

extern "C" int flyhip_bs_sdd_kmajor(const void* a, const void* b, float* c32,
                                    const int32_t* row_ptr, const int32_t* row_blk, const int32_t* row_col,
                                    const int32_t* grp_row0, const int32_t* grp_n, int n_grp, int max_row_nnz,
                                    int brows_per_head, int nnz, int Z, int K, int k_slice, int blk,
                                    int64_t a_sz, int64_t a_sh, int64_t a_sk,
                                    int64_t b_sz, int64_t b_sh, int64_t b_sk,
                                    int dtype, void* stream) {
    int rc = check_common("bs_sdd_kmajor", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(a && b && c32 && row_ptr && row_blk && row_col && grp_row0 && grp_n, "bs_sdd_kmajor: null pointer");
    FLY_REQUIRE(blk == 32 && (dtype == BF16 || dtype == F16), "bs_sdd_kmajor: needs 32x32 blocks of bf16 / fp16");
    FLY_REQUIRE(n_grp > 0 && max_row_nnz > 0 && brows_per_head > 0 && nnz > 0 && K > 0, "bs_sdd_kmajor: bad sizes");
    FLY_REQUIRE(k_slice >= 0 && k_slice % 32 == 0, "bs_sdd_kmajor: k_slice must be a multiple of 32 (0: chosen here)");
    FLY_REQUIRE(((a_sz | a_sh | a_sk | b_sz | b_sh | b_sk) % 8) == 0, "bs_sdd_kmajor: strides must be multiples of 8 elements");
    FLY_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) % 16) == 0, "bs_sdd_kmajor: operands must be 16-byte aligned");
    const Machine& mach = machine();
    const int pairs = (max_row_nnz + 1) / 2, chunks = (pairs + SDDK_MAX_PAIRS - 1) / SDDK_MAX_PAIRS;
    const int np = std::max(2, (pairs + chunks - 1) / chunks);
    if (k_slice == 0) {
        // the slice length that minimises (rounds of workgroups, one per compute unit) x (steps of a slice + the dozen that
        // filling the stages and the atomics cost)
        const long tiles = (long)n_grp * chunks * Z;
        long best = -1;
        for (int n = 1; n <= std::max(1, K / 64) && (n == 1 || tiles * (n - 1) < 4L * mach.cus); ++n) {
            const int steps = ((K + n - 1) / n + 31) / 32;
            const long cost = ((tiles * n + mach.cus - 1) / mach.cus) * (steps + 12);
            if (best < 0 || cost < best) { best = cost; k_slice = 32 * steps; }
        }
    }
    const int slices = (K + k_slice - 1) / k_slice;
    const long items = (long)n_grp * chunks * slices;
    FLY_REQUIRE(items <= 2147483647L - 64, "bs_sdd_kmajor: too many workgroups");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    SddKArgs args{a, b, c32, row_ptr, row_blk, row_col, grp_row0, grp_n, brows_per_head, K, k_slice, chunks, nnz,
                  a_sz, a_sh, a_sk, b_sz, b_sh, b_sk, n_grp, slices, mach.xcds};
    dim3 grid((unsigned)((items + mach.xcds - 1) / mach.xcds * mach.xcds), 1, Z);
#define SDDK_LAUNCH(TT, NP)                                                                                        \
    {                                                                                                              \
        auto kern = bs_sdd32k_kernel<TT, NP>;                                                                      \
        constexpr size_t smem = (size_t)SDDK_STAGES * sddk_stage_bytes(NP);                                        \
        static std::atomic<unsigned long long> lds_set{0};                                                         \
        if (int rc2 = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "bs_sdd_kmajor")) return rc2; \
        hipLaunchKernelGGL(kern, grid, dim3(512), smem, st, args);                                                 \
    }
#define SDDK_PAIRS(TT)                                                                                             \
    {                                                                                                              \
        if (np == 2) SDDK_LAUNCH(TT, 2) else if (np == 3) SDDK_LAUNCH(TT, 3)                                       \
        else if (np == 4) SDDK_LAUNCH(TT, 4) else SDDK_LAUNCH(TT, 5)                                               \
    }
    if (dtype == BF16) SDDK_PAIRS(bf16_t) else SDDK_PAIRS(f16_t)
#undef SDDK_PAIRS
#undef SDDK_LAUNCH
    return check_launch("bs_sdd32k_kernel");
}

extern "C" int flyhip_bs_dsd(const void* a_sp, const void* b, void* c,
                             const int32_t* seg_ptr, const int32_t* seg_blk, const int32_t* seg_inner,
                             const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                             int n_seg, int rows_per_head, int Z, int N, int blk, int trans_a,
                             int64_t a_sz,
                             int64_t b_sz, int64_t b_sh, int64_t b_sk, int64_t b_sn,
                             int64_t c_sz, int64_t c_sh, int64_t c_sm, int64_t c_sn,
                             int dtype, void* stream) {
    int rc = check_common("bs_dsd", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(a_sp && b && c && seg_ptr && seg_blk && seg_inner, "bs_dsd: null pointer");
    FLY_REQUIRE(n_seg > 0 && rows_per_head > 0 && n_seg % rows_per_head == 0, "bs_dsd: bad segment counts");
    FLY_REQUIRE(N > 0, "bs_dsd: N must be positive");
    if (b_sk == 1) FLY_REQUIRE(((b_sz | b_sh | b_sn) % 4) == 0, "bs_dsd: B strides must be multiples of 4 elements");
    if (c_sn == 1) FLY_REQUIRE(((c_sz | c_sh | c_sm) % 4) == 0, "bs_dsd: C strides must be multiples of 4 elements");
    FLY_REQUIRE(a_sz % 4 == 0, "bs_dsd: sparse batch stride must be a multiple of 4 elements");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    DxdArgs args{a_sp, b, c, seg_ptr, seg_blk, seg_inner, n_seg, rows_per_head, N, trans_a,
                 a_sz, b_sz, b_sh, b_sk, b_sn, c_sz, c_sh, c_sm, c_sn, Z};
    if (blk == 32 && (dtype == BF16 || dtype == F16) && (!trans_a || (uni_ptr && uni_inner && uni_blk)) && b_sn == 1 &&
        c_sn == 1 && N % 8 == 0 &&
        ((a_sz | b_sz | b_sh | b_sk | c_sz | c_sh | c_sm) % 8) == 0) {
        if (uni_ptr && uni_inner && uni_blk) {
            const int gph = (rows_per_head + 3) / 4, n_heads = n_seg / rows_per_head;
            DsdUniArgs ua{a_sp, b, c, uni_ptr, uni_inner, uni_blk, rows_per_head, gph, n_heads, Z, N,
                          a_sz, b_sz, b_sh, b_sk, c_sz, c_sh, c_sm};
            const long nwg = unit_grid((long)n_heads * Z, (long)gph * ((N + 63) / 64));
            ua.n_xcd = machine().xcds;
            FLY_REQUIRE(nwg <= 2147483647L, "bs_dsd: too many workgroups");
            dim3 grid((unsigned)nwg);
            if (dtype == BF16) {
                if (trans_a) hipLaunchKernelGGL((bs_dsd32u_kernel<bf16_t, true>), grid, dim3(256), 0, st, ua);
                else hipLaunchKernelGGL((bs_dsd32u_kernel<bf16_t, false>), grid, dim3(256), 0, st, ua);
            } else {
                if (trans_a) hipLaunchKernelGGL((bs_dsd32u_kernel<f16_t, true>), grid, dim3(256), 0, st, ua);
                else hipLaunchKernelGGL((bs_dsd32u_kernel<f16_t, false>), grid, dim3(256), 0, st, ua);
            }
            return check_launch("bs_dsd32u_kernel");
        }
        const long nwg = unit_grid((long)(n_seg / rows_per_head) * Z, (long)rows_per_head * ((N + 63) / 64));
        args.n_xcd = machine().xcds;
        FLY_REQUIRE(nwg <= 2147483647L, "bs_dsd: too many workgroups");
        dim3 grid((unsigned)nwg);
        if (dtype == BF16) hipLaunchKernelGGL((bs_dsd32_kernel<bf16_t>), grid, dim3(256), 0, st, args);
        else hipLaunchKernelGGL((bs_dsd32_kernel<f16_t>), grid, dim3(256), 0, st, args);
        return check_launch("bs_dsd32_kernel");
    }
    const int tile = blk >= 32 ? 32 : 16;
    const long nblocks = waves_to_blocks((long)n_seg * (blk / tile) * ((N + 31) / 32));
    FLY_REQUIRE(nblocks <= 2147483647L, "bs_dsd: too many blocks");
    dim3 grid((unsigned)nblocks, Z);
    BS_DISPATCH(bs_dsd_kernel, grid, args)
    return check_launch("bs_dsd_kernel");
}

extern "C" int flyhip_bs_dds_bias(const void* a, const void* b_sp, const void* bias, void* c,
                             const int32_t* seg_ptr, const int32_t* seg_blk, const int32_t* seg_inner,
                             const int32_t* grp_row0, const int32_t* grp_n, int n_grp, int max_seg_len,
                             int n_seg, int cols_per_head, int Z, int M, int blk, int trans_b,
                             int64_t a_sz, int64_t a_sh, int64_t a_sm, int64_t a_sk,
                             int64_t b_sz,
                             int64_t c_sz, int64_t c_sh, int64_t c_sm, int64_t c_sn,
                             int dtype, void* stream) {
    int rc = check_common("bs_dds", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(a && b_sp && c && seg_ptr && seg_blk && seg_inner, "bs_dds: null pointer");
    FLY_REQUIRE(n_seg > 0 && cols_per_head > 0 && n_seg % cols_per_head == 0, "bs_dds: bad segment counts");
    FLY_REQUIRE(M > 0, "bs_dds: M must be positive");
    if (a_sk == 1) FLY_REQUIRE(((a_sz | a_sh | a_sm) % 4) == 0, "bs_dds: A strides must be multiples of 4 elements");
    if (c_sn == 1) FLY_REQUIRE(((c_sz | c_sh | c_sm) % 4) == 0, "bs_dds: C strides must be multiples of 4 elements");
    FLY_REQUIRE(b_sz % 4 == 0, "bs_dds: sparse batch stride must be a multiple of 4 elements");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    if (grp_row0 && grp_n && n_grp > 0 && max_seg_len >= 0 && max_seg_len <= DDS_MAX_STEPS && blk == 32 &&
        (dtype == BF16 || dtype == F16) && a_sk == 1 && (long)M * a_sm * 2 < (1L << 32) &&
        c_sn == 1 && ((a_sz | a_sh | a_sm | b_sz | c_sz | c_sh | c_sm) % 8) == 0 && (M + 127) / 128 <= 65535) {
        DdsGroupArgs ga{b_sp, a, c, seg_ptr, seg_blk, seg_inner, grp_row0, grp_n, cols_per_head, M,
                        b_sz, a_sz, a_sh, a_sm, c_sz, c_sh, c_sm};
        const Machine& mach = machine();
        ga.n_xcd = mach.xcds;
        ga.n_grp = n_grp;
        ga.bias = bias;
        // few tokens: 32 tokens of one block-row per workgroup while those are at most two per compute unit.  Measured (us,
        // this / the 128-token tiles): 24 block-rows of 36 blocks, 196 tokens (168 workgroups) 7.6 / 20.2; 24 of 9 blocks,
        // 300 tokens (240) 7.1 / 11.2; transposed, 32 of 48, 400 tokens (416) 20 / 30; past the line 96 of 9 blocks, 196 tokens
        // (672) 12.3 / 11.7; transposed, 32 of 48, 784 tokens (800) 37 / 31
        if ((long)n_seg * ((M + 31) / 32) * Z <= 2L * mach.cus) {
            dim3 grid((unsigned)n_seg, (unsigned)((M + 31) / 32), Z);
            if (dtype == BF16) {
                if (trans_b) hipLaunchKernelGGL((bs_dds32w_kernel<bf16_t, false>), grid, dim3(512), 0, st, ga);
                else hipLaunchKernelGGL((bs_dds32w_kernel<bf16_t, true>), grid, dim3(512), 0, st, ga);
            } else {
                if (trans_b) hipLaunchKernelGGL((bs_dds32w_kernel<f16_t, false>), grid, dim3(512), 0, st, ga);
                else hipLaunchKernelGGL((bs_dds32w_kernel<f16_t, true>), grid, dim3(512), 0, st, ga);
            }
            return check_launch("bs_dds32w_kernel");
        }
        // groups whose weights fit the LDS (four output blocks times the longest reduction list) and enough tokens to
        // amortise bringing them in: the weight-stationary kernel, two workgroups per compute unit
        if (FLY_DDS_STATIONARY == 2 && max_seg_len > 0 && max_seg_len <= DDS_STAT_STEPS && (long)M >= 512L * 8) {
            // one workgroup of eight waves per compute unit: the group's weights and a stage of activations per wave
            // streams of token tiles per group: the count that minimises (rounds of workgroups) x (tiles per workgroup)
            const long tiles = (M + 511) / 512;
            long n_streams = 1, best = -1;
            for (long n = 1; n <= tiles && n * n_grp * Z <= 4L * mach.cus + (long)n_grp * Z; ++n) {
                const long cost = ((n * n_grp * Z + mach.cus - 1) / mach.cus) * ((tiles + n - 1) / n);
                if (best < 0 || cost < best) { best = cost; n_streams = n; }
            }
            const long pairs = n_streams * n_grp;
            const long gx = (pairs + mach.xcds - 1) / mach.xcds * mach.xcds;
            const size_t smem = (size_t)DDS_STAT_STEPS * 8192 + 8 * 8192;
            dim3 grid((unsigned)gx, Z);
#define DDS_DMA(TT, WTT)                                                                                           \
    {                                                                                                              \
        auto kern = bs_dds32d_kernel<TT, WTT>;                                                                     \
        static std::atomic<unsigned long long> lds_set{0};                                                         \
        if (int rc2 = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "bs_dds (staged)")) return rc2; \
        hipLaunchKernelGGL(kern, grid, dim3(512), smem, st, ga, (int)n_streams);                                   \
    }
            if (dtype == BF16) { if (trans_b) DDS_DMA(bf16_t, false) else DDS_DMA(bf16_t, true) }
            else { if (trans_b) DDS_DMA(f16_t, false) else DDS_DMA(f16_t, true) }
#undef DDS_DMA
            return check_launch("bs_dds32d_kernel");
        }
        if (FLY_DDS_STATIONARY == 2 && max_seg_len > DDS_STAT_STEPS && max_seg_len <= DDS_MAX_STEPS && (long)M >= 512L * 8 &&
            (trans_b || !bias) && reinterpret_cast<uintptr_t>(b_sp) % 16 == 0) {
            // longer lists: the same workgroup shape with the weights passing through LDS, by transfers of 16 bytes that have to start
            // at a multiple of that ([k][n] blocks: no bias)
            const long tiles = (M + 511) / 512;
            long n_streams = 1, best = -1;
            for (long n = 1; n <= tiles && n * n_grp * Z <= 4L * mach.cus + (long)n_grp * Z; ++n) {
                const long cost = ((n * n_grp * Z + mach.cus - 1) / mach.cus) * ((tiles + n - 1) / n);
                if (best < 0 || cost < best) { best = cost; n_streams = n; }
            }
            const long pairs = n_streams * n_grp;
            const long gx = (pairs + mach.xcds - 1) / mach.xcds * mach.xcds;
            const size_t smem = DDS_PIPE_LDS;
            dim3 grid((unsigned)gx, Z);
#define DDS_CHUNKED(TT, WTT)                                                                                       \
    {                                                                                                              \
        auto kern = bs_dds32c_kernel<TT, WTT>;                                                                     \
        static std::atomic<unsigned long long> lds_set{0};                                                         \
        if (int rc2 = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "bs_dds (chunked)")) return rc2; \
        hipLaunchKernelGGL(kern, grid, dim3(512), smem, st, ga, (int)n_streams);                                   \
    }
            if (dtype == BF16) { if (trans_b) DDS_CHUNKED(bf16_t, false) else DDS_CHUNKED(bf16_t, true) }
            else { if (trans_b) DDS_CHUNKED(f16_t, false) else DDS_CHUNKED(f16_t, true) }
#undef DDS_CHUNKED
            return check_launch("bs_dds32c_kernel");
        }
        if (FLY_DDS_STATIONARY && max_seg_len > 0 && max_seg_len <= DDS_STAT_STEPS && (long)M >= 256L * 8) {
            const long tiles = (M + 255) / 256;
            long n_streams = 2L * mach.cus / ((long)n_grp * Z);
            if (n_streams < 1) n_streams = 1;
            if (n_streams > tiles) n_streams = tiles;
            const long pairs = n_streams * n_grp;
            const long gx = (pairs + mach.xcds - 1) / mach.xcds * mach.xcds;
            const size_t smem = (size_t)max_seg_len * 8192;
            dim3 grid((unsigned)gx, Z);
#define DDS_STAT(TT, WTT)                                                                                          \
    {                                                                                                              \
        auto kern = bs_dds32s_kernel<TT, WTT, FLY_DDS_DEPTH>;                                                       \
        static std::atomic<unsigned long long> lds_set{0};                                                         \
        if (int rc2 = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_set, "bs_dds (stationary)")) return rc2; \
        hipLaunchKernelGGL(kern, grid, dim3(256), smem, st, ga, (int)n_streams);                                   \
    }
            if (dtype == BF16) { if (trans_b) DDS_STAT(bf16_t, false) else DDS_STAT(bf16_t, true) }
            else { if (trans_b) DDS_STAT(f16_t, false) else DDS_STAT(f16_t, true) }
#undef DDS_STAT
            return check_launch("bs_dds32s_kernel");
        }
        // as many workgroups as are resident together (two fit a CU: 64 KB of tiles each); each walks its share of the
        // token tiles
        const long tiles = (M + 127) / 128;
        long gy = (2L * mach.cus + (long)n_grp * Z - 1) / ((long)n_grp * Z);
        if (gy > tiles) gy = tiles;
        gy = (gy + mach.xcds - 1) / mach.xcds * mach.xcds;   // the kernel deals streams of token tiles to the XCDs
        dim3 grid(n_grp, (unsigned)gy, Z);
        constexpr size_t smem_t = 4 * 128 * 64 * 2;          // two stages of the activation and the weight tile
#define DDS_TILED(TT, WTT)                                                                                         \
    {                                                                                                              \
        auto kern = bs_dds32_kernel<TT, WTT>;                                                                      \
        static std::atomic<unsigned long long> lds_set{0};                                                         \
        if (int rc2 = ensure_dynamic_lds(reinterpret_cast<const void*>(kern), smem_t, lds_set, "bs_dds (tiled)")) return rc2; \
        hipLaunchKernelGGL(kern, grid, dim3(256), smem_t, st, ga);                                                 \
    }
        if (dtype == BF16) { if (trans_b) DDS_TILED(bf16_t, false) else DDS_TILED(bf16_t, true) }
        else { if (trans_b) DDS_TILED(f16_t, false) else DDS_TILED(f16_t, true) }
#undef DDS_TILED
        return check_launch("bs_dds32_kernel");
    }
    DxdArgs args{b_sp, a, c, seg_ptr, seg_blk, seg_inner, n_seg, cols_per_head, M, trans_b,
                 b_sz, a_sz, a_sh, a_sm, a_sk, c_sz, c_sh, c_sm, c_sn};
    args.bias = bias;
    const int tile = blk >= 32 ? 32 : 16;
    const long nblocks = waves_to_blocks((long)((M + 31) / 32) * n_seg * (blk / tile));
    FLY_REQUIRE(nblocks <= 2147483647L, "bs_dds: too many blocks");
    dim3 grid((unsigned)nblocks, Z);
    BS_DISPATCH(bs_dds_kernel, grid, args)
    return check_launch("bs_dds_kernel");
}

extern "C" int flyhip_bs_dds(const void* a, const void* b_sp, void* c,
                             const int32_t* seg_ptr, const int32_t* seg_blk, const int32_t* seg_inner,
                             const int32_t* grp_row0, const int32_t* grp_n, int n_grp, int max_seg_len,
                             int n_seg, int cols_per_head, int Z, int M, int blk, int trans_b,
                             int64_t a_sz, int64_t a_sh, int64_t a_sm, int64_t a_sk,
                             int64_t b_sz,
                             int64_t c_sz, int64_t c_sh, int64_t c_sm, int64_t c_sn,
                             int dtype, void* stream) {
    return flyhip_bs_dds_bias(a, b_sp, nullptr, c, seg_ptr, seg_blk, seg_inner, grp_row0, grp_n, n_grp, max_seg_len, n_seg,
                              cols_per_head, Z, M, blk, trans_b, a_sz, a_sh, a_sm, a_sk, b_sz, c_sz, c_sh, c_sm, c_sn, dtype, stream);
}

template <typename T>
static int launch_softmax(const RowArgs& args, dim3 grid, int max_elems, hipStream_t st) {
    if (sizeof(T) == 2 && args.blk_shift == 5 && max_elems <= 32 * 4 * 16 && (args.x_sz % 8) == 0) {
        dim3 g2(2 * args.n_brow, grid.y);
        const int slots = (max_elems / 32 + 3) / 4;          // blocks per wave with four waves: sizes the register arrays
#define SM32(N) hipLaunchKernelGGL((bs_softmax32_kernel<T, N, 4>), g2, dim3(256), 0, st, args)
#define SM32W(N) hipLaunchKernelGGL((bs_softmax32_kernel<T, N, 8>), g2, dim3(512), 0, st, args)
        if (slots <= 4) SM32(4); else if (slots <= 8) SM32(8);
        else if (slots <= 10) SM32W(5); else if (slots <= 12) SM32W(6); else if (slots <= 14) SM32W(7);
        else SM32W(8);
#undef SM32W
#undef SM32
        return check_launch("bs_softmax32_kernel");
    }
    if (max_elems <= 64 * 8) hipLaunchKernelGGL((bs_softmax_kernel<T, 8>), grid, dim3(256), 0, st, args);
    else if (max_elems <= 64 * 32) hipLaunchKernelGGL((bs_softmax_kernel<T, 32>), grid, dim3(256), 0, st, args);
    else hipLaunchKernelGGL((bs_softmax_long_kernel<T>), grid, dim3(256), 0, st, args);
    return check_launch("bs_softmax_kernel");
}

static int bs_attn_checked(const void* q, const void* k, const void* v, void* out, float* lse2,
                              const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                              int rows_per_group, const float* key_mask, int64_t key_mask_stride,
                              const float* attn_mask, int64_t attn_mask_stride,
                              int Z, int H, int brows_per_head, int D, int blk,
                              int64_t q_sz, int64_t q_sh, int64_t q_sm,
                              int64_t k_sz, int64_t k_sh, int64_t k_sn,
                              int64_t v_sz, int64_t v_sh, int64_t v_sn,
                              int64_t o_sz, int64_t o_sh, int64_t o_sm,
                              float scale, int dtype, void* stream, DropArgs drop) {
    int rc = check_common("bs_attn", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(q && k && v && out && uni_ptr && uni_inner && uni_blk, "bs_attn: null pointer");
    FLY_REQUIRE(blk == 32 && (dtype == BF16 || dtype == F16), "bs_attn: needs 32x32 blocks of bf16 / fp16 (got block %d, dtype %d)", blk, dtype);
    FLY_REQUIRE(D == 32 || D == 64 || D == 128, "bs_attn: head dim %d not in {32,64,128}", D);
    FLY_REQUIRE(rows_per_group == 4 || rows_per_group == 8, "bs_attn: rows_per_group must be 4 or 8");
    FLY_REQUIRE(H > 0 && brows_per_head > 0, "bs_attn: bad sizes");
    FLY_REQUIRE(((q_sz | q_sh | q_sm | k_sz | k_sh | k_sn | v_sz | v_sh | v_sn) % 8) == 0,
                "bs_attn: q / k / v strides must be multiples of 8 elements");
    FLY_REQUIRE(((o_sz | o_sh | o_sm) % 4) == 0, "bs_attn: out strides must be multiples of 4 elements");
    FLY_REQUIRE(!key_mask || key_mask_stride % 4 == 0, "bs_attn: key mask stride must be a multiple of 4");
    FLY_REQUIRE(!attn_mask || attn_mask_stride % 4 == 0, "bs_attn: attention mask stride must be a multiple of 4");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    const int gph = (brows_per_head + rows_per_group - 1) / rows_per_group;
    AttnArgs args{q, k, v, out, uni_ptr, uni_inner, uni_blk, key_mask, key_mask_stride, brows_per_head, gph, H, Z,
                  q_sz, q_sh, q_sm, k_sz, k_sh, k_sn, v_sz, v_sh, v_sn, o_sz, o_sh, o_sm, scale, lse2};
    args.am = attn_mask;
    args.am_stride = attn_mask_stride;
    const long nwg = unit_grid((long)H * Z, gph);
    args.n_xcd = machine().xcds;
    FLY_REQUIRE(nwg <= 2147483647L, "bs_attn: too many workgroups");
    dim3 grid((unsigned)nwg);
    const bool masked = key_mask != nullptr || attn_mask != nullptr || !(scale > 0.f);
    const bool dropping = drop.thresh != 0u;
    args.drop_seed = drop.seed;
    args.drop_thresh = drop.thresh;
    args.drop_scale = drop.scale;
#define ATTN_LAUNCH(T, KS, NW)                                                                                  \
    do {                                                                                                        \
        if (dropping && masked) hipLaunchKernelGGL((bs_attn32_kernel<T, KS, NW, true, true>), grid, dim3(64 * NW), 0, st, args); \
        else if (dropping) hipLaunchKernelGGL((bs_attn32_kernel<T, KS, NW, false, true>), grid, dim3(64 * NW), 0, st, args); \
        else if (masked) hipLaunchKernelGGL((bs_attn32_kernel<T, KS, NW, true>), grid, dim3(64 * NW), 0, st, args);  \
        else hipLaunchKernelGGL((bs_attn32_kernel<T, KS, NW, false>), grid, dim3(64 * NW), 0, st, args);        \
    } while (0)
#define ATTN_KS(T, NW) do { if (D == 32) ATTN_LAUNCH(T, 1, NW); else if (D == 64) ATTN_LAUNCH(T, 2, NW); else ATTN_LAUNCH(T, 4, NW); } while (0)
    if (dtype == BF16) { if (rows_per_group == 4) ATTN_KS(bf16_t, 4); else ATTN_KS(bf16_t, 8); }
    else { if (rows_per_group == 4) ATTN_KS(f16_t, 4); else ATTN_KS(f16_t, 8); }
#undef ATTN_KS
#undef ATTN_LAUNCH
    return check_launch("bs_attn32_kernel");
}

extern "C" int flyhip_bs_attn_masks(const void* q, const void* k, const void* v, void* out, float* lse2,
                              const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                              int rows_per_group, const float* key_mask, int64_t key_mask_stride,
                              const float* attn_mask, int64_t attn_mask_stride,
                              int Z, int H, int brows_per_head, int D, int blk,
                              int64_t q_sz, int64_t q_sh, int64_t q_sm,
                              int64_t k_sz, int64_t k_sh, int64_t k_sn,
                              int64_t v_sz, int64_t v_sh, int64_t v_sn,
                              int64_t o_sz, int64_t o_sh, int64_t o_sm,
                              float scale, int dtype, void* stream) {
    return bs_attn_checked(q, k, v, out, lse2, uni_ptr, uni_inner, uni_blk, rows_per_group, key_mask, key_mask_stride,
                           attn_mask, attn_mask_stride, Z, H, brows_per_head, D, blk, q_sz, q_sh, q_sm, k_sz, k_sh, k_sn,
                           v_sz, v_sh, v_sn, o_sz, o_sh, o_sm, scale, dtype, stream, DropArgs{0u, 0u, 1.f});
}

extern "C" int flyhip_bs_attn_dropout(const void* q, const void* k, const void* v, void* out, float* lse2,
                              const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                              int rows_per_group, const float* key_mask, int64_t key_mask_stride,
                              const float* attn_mask, int64_t attn_mask_stride,
                              int Z, int H, int brows_per_head, int D, int blk,
                              int64_t q_sz, int64_t q_sh, int64_t q_sm,
                              int64_t k_sz, int64_t k_sh, int64_t k_sn,
                              int64_t v_sz, int64_t v_sh, int64_t v_sn,
                              int64_t o_sz, int64_t o_sh, int64_t o_sm,
                              float scale, int dtype, float dropout_p, uint64_t dropout_seed, void* stream) {
    FLY_REQUIRE(dropout_p >= 0.f && dropout_p < 1.f, "bs_attn_dropout: dropout_p %g not in [0, 1)", (double)dropout_p);
    FLY_REQUIRE((long)Z * H * brows_per_head * 32 <= 4294967295L, "bs_attn_dropout: more than 2^32 rows");
    return bs_attn_checked(q, k, v, out, lse2, uni_ptr, uni_inner, uni_blk, rows_per_group, key_mask, key_mask_stride,
                           attn_mask, attn_mask_stride, Z, H, brows_per_head, D, blk, q_sz, q_sh, q_sm, k_sz, k_sh, k_sn,
                           v_sz, v_sh, v_sn, o_sz, o_sh, o_sm, scale, dtype, stream, drop_args(dropout_p, dropout_seed));
}

extern "C" int flyhip_bs_attn_lse(const void* q, const void* k, const void* v, void* out, float* lse2,
                              const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                              int rows_per_group, const float* key_mask, int64_t key_mask_stride,
                              int Z, int H, int brows_per_head, int D, int blk,
                              int64_t q_sz, int64_t q_sh, int64_t q_sm,
                              int64_t k_sz, int64_t k_sh, int64_t k_sn,
                              int64_t v_sz, int64_t v_sh, int64_t v_sn,
                              int64_t o_sz, int64_t o_sh, int64_t o_sm,
                              float scale, int dtype, void* stream) {
    return flyhip_bs_attn_masks(q, k, v, out, lse2, uni_ptr, uni_inner, uni_blk, rows_per_group, key_mask, key_mask_stride,
                                nullptr, 0, Z, H, brows_per_head, D, blk, q_sz, q_sh, q_sm, k_sz, k_sh, k_sn, v_sz, v_sh, v_sn,
                                o_sz, o_sh, o_sm, scale, dtype, stream);
}

extern "C" int flyhip_bs_attn(const void* q, const void* k, const void* v, void* out,
                              const int32_t* uni_ptr, const int32_t* uni_inner, const int32_t* uni_blk,
                              int rows_per_group, const float* key_mask, int64_t key_mask_stride,
                              int Z, int H, int brows_per_head, int D, int blk,
                              int64_t q_sz, int64_t q_sh, int64_t q_sm,
                              int64_t k_sz, int64_t k_sh, int64_t k_sn,
                              int64_t v_sz, int64_t v_sh, int64_t v_sn,
                              int64_t o_sz, int64_t o_sh, int64_t o_sm,
                              float scale, int dtype, void* stream) {
    return flyhip_bs_attn_lse(q, k, v, out, nullptr, uni_ptr, uni_inner, uni_blk, rows_per_group, key_mask, key_mask_stride,
                              Z, H, brows_per_head, D, blk, q_sz, q_sh, q_sm, k_sz, k_sh, k_sn, v_sz, v_sh, v_sn,
                              o_sz, o_sh, o_sm, scale, dtype, stream);
}

extern "C" int flyhip_bs_softmax(void* x, const int32_t* row_ptr, const int32_t* row_blk, const int32_t* row_col,
                                 int n_brow, int brows_per_head, int max_row_nnz, int Z, int blk, int64_t x_sz,
                                 float scale, const float* kpm, int64_t kpm_stride, int kpm_mul,
                                 const float* am, int64_t am_stride, int am_mul, int dtype, void* stream) {
    int rc = check_common("bs_softmax", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(x && row_ptr && row_blk && row_col, "bs_softmax: null pointer");
    FLY_REQUIRE(n_brow > 0 && brows_per_head > 0 && n_brow % brows_per_head == 0, "bs_softmax: bad row counts");
    FLY_REQUIRE(max_row_nnz >= 0, "bs_softmax: negative max_row_nnz");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    RowArgs args{x, nullptr, row_ptr, row_blk, row_col, n_brow, brows_per_head, blk_shift_of(blk), x_sz, scale,
                 kpm, kpm_stride, kpm_mul, am, am_stride, am_mul, 0};
    const long nblocks = waves_to_blocks((long)n_brow * blk);
    dim3 grid((unsigned)nblocks, Z);
    const int max_elems = max_row_nnz * blk;   // selects the register-resident or the multi-pass kernel
    switch (dtype) {
        case F32: return launch_softmax<float>(args, grid, max_elems, st);
        case BF16: return launch_softmax<bf16_t>(args, grid, max_elems, st);
        default: return launch_softmax<f16_t>(args, grid, max_elems, st);
    }
}

extern "C" int flyhip_bs_softmax_bwd(const void* y, const void* dy, void* dx,
                                     const int32_t* row_ptr, const int32_t* row_blk,
                                     int n_brow, int max_row_nnz, int Z, int blk, int64_t y_sz,
                                     float scale, int dtype, void* stream) {
    int rc = check_common("bs_softmax_bwd", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(y && dy && dx && row_ptr && row_blk, "bs_softmax_bwd: null pointer");
    FLY_REQUIRE(blk == 32 && (dtype == BF16 || dtype == F16), "bs_softmax_bwd: needs 32x32 blocks of bf16 / fp16");
    FLY_REQUIRE(n_brow > 0 && max_row_nnz >= 0 && max_row_nnz <= 64, "bs_softmax_bwd: at most 64 blocks per block-row (got %d)", max_row_nnz);
    FLY_REQUIRE(y_sz % 8 == 0, "bs_softmax_bwd: batch stride must be a multiple of 8 elements");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    RowBwdArgs args{y, dy, dx, row_ptr, row_blk, y_sz, scale};
    dim3 grid(2 * n_brow, Z);
    const int slots = (max_row_nnz + 3) / 4;
#define SMB(T, N) hipLaunchKernelGGL((bs_softmax32_bwd_kernel<T, N, 4>), grid, dim3(256), 0, st, args)
    // (four waves measured faster than eight here -- 0.68 against 0.77 ms at config 2 -- the opposite of the forward kernel)
#define SMB_T(T) do { if (slots <= 4) SMB(T, 4); else if (slots <= 8) SMB(T, 8); else if (slots <= 13) SMB(T, 13); else SMB(T, 16); } while (0)
    if (dtype == BF16) SMB_T(bf16_t); else SMB_T(f16_t);
#undef SMB_T
#undef SMB
    return check_launch("bs_softmax32_bwd_kernel");
}

extern "C" int flyhip_bs_rowreduce(const void* x, void* out, const int32_t* row_ptr, const int32_t* row_blk,
                                   int n_brow, int Z, int blk, int64_t x_sz, int op, int dtype, void* stream) {
    int rc = check_common("bs_rowreduce", blk, dtype, Z);
    if (rc) return rc;
    FLY_REQUIRE(x && out && row_ptr && row_blk, "bs_rowreduce: null pointer");
    FLY_REQUIRE(op == 0 || op == 1, "bs_rowreduce: op must be 0 (logsumexp) or 1 (sum)");
    FLY_REQUIRE(n_brow > 0, "bs_rowreduce: no rows");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (int rc_capture = refuse_capture(st)) return rc_capture;
    RowArgs args{const_cast<void*>(x), out, row_ptr, row_blk, nullptr, n_brow, 1, blk_shift_of(blk), x_sz, 1.f,
                 nullptr, 0, 0, nullptr, 0, 0, op};
    dim3 grid((unsigned)waves_to_blocks((long)n_brow * blk), Z);
    switch (dtype) {
        case F32: hipLaunchKernelGGL((bs_rowreduce_kernel<float>), grid, dim3(256), 0, st, args); break;
        case BF16: hipLaunchKernelGGL((bs_rowreduce_kernel<bf16_t>), grid, dim3(256), 0, st, args); break;
        default: hipLaunchKernelGGL((bs_rowreduce_kernel<f16_t>), grid, dim3(256), 0, st, args); break;
    }
    return check_launch("bs_rowreduce_kernel");
}
