// Attention forward and backward for fp32 tensors on the fp32 matrix instructions
// (v_mfma_f32_16x16x4_f32: fp32 operands, fp32 products and sums -- no reduced-precision input
// anywhere), the kernels behind dtype == SLAPO_F32, whose parity bar is 1e-5 absolute.
//
// v_mfma_f32_16x16x4_f32 (one wavefront, lane l, i = l % 16, g = l / 16):
//   A operand: lane holds A[row i][k-slot g];   B operand: lane holds B[k-slot g][column i];
//   C/D:       register r of lane l is element (row 4 g + r, column i).
// The k-slots may stand for any data as long as A and B agree.  Two choices keep every operand a
// plain LDS read or a register:
//  * products over the head dimension (S = QK^T, dP = dO V^T): slot g of step 4 t + e is element
//    16 t + 4 g + e, so that one 16-byte read of a row serves four steps;
//  * products over keys or queries (PV, dS K, P^T dO, dS^T Q): an accumulator register r of the
//    previous product holds row 4 g + r of its column -- exactly slot g of step r -- so
//    probabilities never leave registers, and the other operand is row 4 g + r of the row-major
//    tile in LDS, sixteen lanes on consecutive elements.
// With a row pitch of 16 DB + 4 floats both access patterns touch all 64 banks once.
//
// One workgroup = 4 wavefronts x 16 rows (queries in forward and dQ, keys in dK/dV); the other side
// streams through LDS in tiles of 32 rows, double buffered, staged through registers.  Bound by the
// matrix pipe: 256 FLOP per cycle and CU (157 TFLOP/s nominal; a large fp32 library product reaches
// 138 on this card).  A wavefront spends 32 DB x 16 matrix cycles per tile and product against about
// 200 vector instructions, and needs few registers, so several wavefronts share a SIMD and hide each
// other's vector work.  B4 S512 H16 D64 without a mask, forward: 51.5 us = 83 TFLOP/s (one thread per row
// on plain FMAs: 686 us, 6.3 TFLOP/s); B2 S2048 H16 D128 696 us = 99 TFLOP/s.
//
// Reference semantics: slapo/op/attention.py:163-181 (attention_bmk) and its autograd.
#include "attn_common.h"

using namespace slapo;

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kRows = kWaves * 16;  // rows owned by a workgroup
constexpr int kTile = 32;           // streamed rows per LDS tile
// Forward calls that give a CU two workgroups at most run kHalves = 2: eight wavefronts, two per 16
// query rows, each with one half of a tile of 64 keys and a softmax state of its own, merged at the end
// through LDS.  Four wavefronts per SIMD then hide the vector work of a launch that has no more rows
// (B4 S512 H16 D64 56.6 -> 51.5 us, D80 83.7 -> 72.6, B1 S4096 H2 D64 causal 113 -> 102); with more
// workgroups the other ones do that and the merge only costs (B16 S512 H16 D64 184 -> 191 us, B2 S2048
// H16 D128 696 -> 750).
constexpr int64_t kHalvesBlocks = 512;  // two for each of 256 CUs

__device__ __forceinline__ f32x4_t mma(float a, float b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// Across the four lanes that share a column (l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ float column_max(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float column_sum(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

__device__ __forceinline__ float bias_at(const AttnArgs& a, int b, int h, int i, int j) {
    return canonical_bias(bias_load(
        a, b * a.bs[0] + h * a.bs[1] + (int64_t)i * a.bs[2] + (int64_t)j * a.bs[3]));
}

// LDS row pitch of a tile, in floats
template <int DB>
constexpr int kPitchOf = 16 * DB + 4;

// Builds of each kernel: kMode & 1 = with a bias, kMode & 2 = with dropout, for tensors whose rows are
// 16-byte aligned with d % 4 == 0; kGeneral serves every other layout element by element and decides
// about bias and dropout when it runs.
constexpr int kGeneral = 4;

// A tile of kTileRows rows of 16 DB floats on its way from global memory to LDS.  Rows past the end are
// clamped, columns past d read as zero.
template <int DB, bool kVec, int kTileRows = kTile, int kBlock = kThreads>
struct Tile {
    static constexpr int kPitch = kPitchOf<DB>;
    static constexpr int kElems = kTileRows * kPitch;
    static constexpr int kPerRow = 4 * DB;
    static constexpr int kChunks = kTileRows * kPerRow;
    static constexpr int kPer = (kChunks + kBlock - 1) / kBlock;
    f32x4_t r[kPer];

    __device__ __forceinline__ void load(const float* base, int64_t stride, int row0, int n_rows,
                                         int d) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = threadIdx.x + u * kBlock;
            if (kChunks % kBlock != 0 && c >= kChunks) continue;
            const float* row = base + (int64_t)min(row0 + c / kPerRow, n_rows - 1) * stride;
            const int col = 4 * (c % kPerRow);
            if constexpr (kVec) {
                r[u] = *reinterpret_cast<const f32x4_t*>(row + min(col, d - 4));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) r[u][e] = row[min(col + e, d - 1)];
            }
        }
    }
    __device__ __forceinline__ void store(float* lds, int row0, int n_rows, int d) const {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = threadIdx.x + u * kBlock;
            if (kChunks % kBlock != 0 && c >= kChunks) continue;
            const int row = c / kPerRow, col = 4 * (c % kPerRow);
            f32x4_t v = r[u];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row0 + row >= n_rows || col + e >= d) v[e] = 0.f;
            *reinterpret_cast<f32x4_t*>(lds + row * kPitch + col) = v;
        }
    }
};

// Register fragments of row `row` (16 DB elements, 4 per step group): element 16 t + 4 g + e.
template <bool kVec, int DB>
__device__ __forceinline__ void load_frags(f32x4_t (&f)[DB], const float* base, int64_t stride,
                                           int row, int n_rows, int d, float scale) {
    const int g = (threadIdx.x & 63) >> 4;
    const float* p = base + (int64_t)min(row, n_rows - 1) * stride;
#pragma unroll
    for (int t = 0; t < DB; ++t) {
        const int col = 16 * t + 4 * g;
        if constexpr (kVec) {
            f[t] = *reinterpret_cast<const f32x4_t*>(p + min(col, d - 4));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[t][e] = p[min(col + e, d - 1)];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            f[t][e] = (row < n_rows && col + e < d) ? f[t][e] * scale : 0.f;
    }
}

// c += A B over the head dimension: A = 16 tile rows from row `r0` on, B = this lane's fragments.
template <int DB>
__device__ __forceinline__ f32x4_t dot_rows(const float* tile, int r0, const f32x4_t (&f)[DB]) {
    const int lane = threadIdx.x & 63;
    const float* p = tile + (r0 + (lane & 15)) * kPitchOf<DB> + 4 * (lane >> 4);
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DB; ++t) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(p + 16 * t);
#pragma unroll
        for (int e = 0; e < 4; ++e) c = mma(v[e], f[t][e], c);
    }
    return c;
}
// acc[x] += A B over the 16 tile rows from r0 on: A = columns 16 x .. 16 x + 15 of those rows
// (transposed), B = w, register r of it being row 4 g + r of this lane's column.
template <int DB>
__device__ __forceinline__ void add_rows(const float* tile, int r0, const f32x4_t& w,
                                         f32x4_t (&acc)[DB]) {
    const int lane = threadIdx.x & 63;
    const float* p = tile + (r0 + 4 * (lane >> 4)) * kPitchOf<DB> + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int x = 0; x < DB; ++x) acc[x] = mma(p[r * kPitchOf<DB> + 16 * x], w[r], acc[x]);
}

// Writes this lane's column of acc (element 16 x + 4 g + r in acc[x][r]) times mul as row `row`.
template <bool kVec, int DB>
__device__ __forceinline__ void store_row(const f32x4_t (&acc)[DB], float mul, float* row, int d) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int x = 0; x < DB; ++x) {
        const int col = 16 * x + 4 * g;
        if constexpr (kVec) {
            if (col < d) *reinterpret_cast<f32x4_t*>(row + col) = acc[x] * mul;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < d) row[col + e] = acc[x][e] * mul;
        }
    }
}

// Keep bits (bit r: key j + r) of query i and the four keys from j on, j % 4 == 0.
__device__ __forceinline__ uint32_t keep_keys(const AttnArgs& a, int bh, int i, int j) {
    const uint64_t e = ((uint64_t)bh * a.sq + (uint64_t)i) * (uint64_t)a.sk + (uint64_t)j;
    if (i >= a.sq || j >= a.sk) return 0;
    if (a.dropout == 1) return dropout_keep4_pow2(a.rng, e >> 2);
    return dropout_keep_any(a.rng, e, min(4, a.sk - j));
}
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xF, 0xF, false);
}
// The same for a lane whose registers are the queries i .. i + 3 and whose key is j0 + l % 16 (bit
// r: query i + r): a Philox block covers four consecutive keys, i.e. the four lanes of a quad, so
// lane c of a quad draws the block of query i + c and the quad exchanges them.
__device__ __forceinline__ uint32_t keep_queries(const AttnArgs& a, int bh, int i, int j0) {
    const int c = threadIdx.x & 3, j = j0 + (threadIdx.x & 15);
    const uint32_t mine = keep_keys(a, bh, i + c, j - c);
    return ((dpp<0x00>(mine) >> c) & 1u) | (((dpp<0x55>(mine) >> c) & 1u) << 1) |
           (((dpp<0xAA>(mine) >> c) & 1u) << 2) | (((dpp<0xFF>(mine) >> c) & 1u) << 3);
}

// What a workgroup of the query-owning kernels works on: heaviest query tiles first, the heads as
// the fast index so that the tiles of one head share an XCD's L2.
struct Place {
    int b, h, bh, row0, split;
    int64_t part_row0;  // of the split's partial result, rows of all (batch, head) pairs
    __device__ __forceinline__ Place(const AttnArgs& a, int n_rows, bool last_first) {
        const int n_bh = a.batch * a.heads;
        const int n_t = (n_rows + kRows - 1) / kRows;
        bh = (int)(blockIdx.x % (unsigned)n_bh);
        int t = (int)(blockIdx.x / (unsigned)n_bh);
        split = t / n_t;
        t -= split * n_t;
        part_row0 = ((int64_t)split * n_bh + bh) * n_rows;
        b = bh / a.heads, h = bh % a.heads;
        row0 = (last_first ? n_t - 1 - t : t) * kRows;
    }
};

// Which elements c of a lane's run are visible: lo <= c <= hi.
struct Visible {
    int lo, hi;
    __device__ __forceinline__ bool operator()(int c) const { return c >= lo && c <= hi; }
};
// the run starts at key `first` of query i
__device__ __forceinline__ Visible keys_of_query(const AttnArgs& a, int i, int first, bool masked) {
    if (!masked) return {0, kTile};
    return {(a.window > 0 ? i - a.window + 1 : 0) - first,
            (a.causal ? min(i, a.sk - 1) : a.sk - 1) - first};
}
// the run starts at query `first` of key j
__device__ __forceinline__ Visible queries_of_key(const AttnArgs& a, int j, int first,
                                                  bool masked) {
    if (!masked) return {0, kTile};
    return {(a.causal ? j : 0) - first,
            (a.window > 0 ? min(j + a.window, a.sq) - 1 : a.sq - 1) - first};
}

template <int DB, int kMode, int kHalves>
__global__ __launch_bounds__(kHalves* kThreads, DB <= 4 ? kHalves + 2 : 2) void attn_f32_fwd_kernel(
    const AttnArgs a_in) {
    constexpr int kFwdThreads = kHalves * kThreads, kFwdTile = kHalves * kTile;
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    if (dropout) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    typedef Tile<DB, kVec, kFwdTile, kFwdThreads> tile_t;
    constexpr int kElems = tile_t::kElems;
    float* ks = lds;               // K[2][tile]
    float* vs = lds + 2 * kElems;  // V[2][tile]
    const Place at(a, a.sq, true);
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wq0 = at.row0 + 16 * (wave % kWaves);
    const int half = wave / kWaves;  // of every tile's keys
    const int i = wq0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];

    int j_lo, j_hi;
    key_range(a, at.row0, min(at.row0 + kRows, a.sq), j_lo, j_hi);
    j_hi = max(j_lo + 1, min(j_hi, has_bias ? padded_key_limit<kFwdThreads, true>(a, at.b, at.h, lds) : a.sk));
    int t_lo = j_lo / kFwdTile, t_hi = (j_hi + kFwdTile - 1) / kFwdTile;
    if (a.n_split > 1) split_tiles(a, at.split, t_lo, t_hi);

    tile_t kt, vt;
    f32x4_t qf[DB], o[DB];
    kt.load(kp, a.ks[1], t_lo * kFwdTile, a.sk, a.d);
    vt.load(vp, a.vs[1], t_lo * kFwdTile, a.sk, a.d);
    load_frags<kVec>(qf, qp, a.qs[1], i, a.sq, a.d, a.scale);
#pragma unroll
    for (int x = 0; x < DB; ++x) o[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;  // l: this lane's share of the row sum
    kt.store(ks, t_lo * kFwdTile, a.sk, a.d);
    vt.store(vs, t_lo * kFwdTile, a.sk, a.d);
    __syncthreads();

    const int wq_last = min(wq0 + 15, a.sq - 1);
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const int part = half * kTile * tile_t::kPitch;
        const float *kb = ks + slot * kElems + part, *vb = vs + slot * kElems + part;
        if (t + 1 < t_hi) {
            kt.load(kp, a.ks[1], (t + 1) * kFwdTile, a.sk, a.d);
            vt.load(vp, a.vs[1], (t + 1) * kFwdTile, a.sk, a.d);
        }
        const int j0 = t * kFwdTile + half * kTile;
        const bool active = wq0 < a.sq && j0 < a.sk && (!a.causal || j0 <= wq_last) &&
                            (a.window <= 0 || wq0 - (j0 + kTile - 1) < a.window);
        if (active) {  // uniform per wavefront
            f32x4_t s[2];
            s[0] = dot_rows<DB>(kb, 0, qf);
            s[1] = dot_rows<DB>(kb, 16, qf);
            const bool masked = j0 + kTile > a.sk || (a.causal && j0 + kTile - 1 > wq0) ||
                                (a.window > 0 && wq_last - j0 >= a.window);
            const Visible vis = keys_of_query(a, i, j0 + 4 * g, masked);
            float mx = -INFINITY;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = j0 + 16 * h2 + 4 * g + r;
                    if (has_bias)
                        s[h2][r] += bias_at(a, at.b, at.h, min(i, a.sq - 1), min(j, a.sk - 1));
                    s[h2][r] = vis(16 * h2 + r) ? s[h2][r] : -INFINITY;
                    mx = fmaxf(mx, s[h2][r]);
                }
            const float m_new = fmaxf(m, column_max(mx));
            if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {
                const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int x = 0; x < DB; ++x) o[x] *= alpha;
            }
            const float m_ref = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                uint32_t bits = 0xFu;
                if (dropout) bits = keep_keys(a, at.bh, i, j0 + 16 * h2 + 4 * g);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float p = expf(s[h2][r] - m_ref);
                    l += p;
                    if (dropout) p = (bits >> r) & 1u ? p * a.rng.inv_keep : 0.f;
                    s[h2][r] = p;
                }
                add_rows<DB>(vb, 16 * h2, s[h2], o);
            }
        }
        if (t + 1 < t_hi) {
            kt.store(ks + (slot ^ 1) * kElems, (t + 1) * kFwdTile, a.sk, a.d);
            vt.store(vs + (slot ^ 1) * kElems, (t + 1) * kFwdTile, a.sk, a.d);
        }
        __syncthreads();
    }
    float l_tot = column_sum(l);
    if constexpr (kHalves == 2) {
        // the second half's state joins the first's through LDS (every wavefront is past the loop's
        // last barrier): lane by lane, the two hold the same rows and columns
        float* state = lds + (wave % kWaves) * (4 * DB + 2) * 64 + lane;
        if (half != 0) {
#pragma unroll
            for (int x = 0; x < DB; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) state[(4 * x + e) * 64] = o[x][e];
            state[4 * DB * 64] = m, state[(4 * DB + 1) * 64] = l_tot;
        }
        __syncthreads();
        if (half != 0) return;
        const float m2 = state[4 * DB * 64], m_all = fmaxf(m, m2);
        const float w1 = m == -INFINITY ? 0.f : expf(m - m_all);
        const float w2 = m2 == -INFINITY ? 0.f : expf(m2 - m_all);
        l_tot = l_tot * w1 + state[(4 * DB + 1) * 64] * w2;
        m = m_all;
#pragma unroll
        for (int x = 0; x < DB; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[x][e] = o[x][e] * w1 + state[(4 * x + e) * 64] * w2;
    }
    if (i >= a.sq) return;
    if (a.n_split > 1) {
        store_row<kVec>(o, 1.0f, a.part + (at.part_row0 + i) * a.d, a.d);
        if (g == 0) {
            float* ml = a.part + (int64_t)a.n_split * a.batch * a.heads * a.sq * a.d +
                        2 * (at.part_row0 + i);
            ml[0] = m, ml[1] = l_tot;
        }
        return;
    }
    float* op = reinterpret_cast<float*>(a.o) + at.b * a.os[0] + (int64_t)i * a.os[1] +
                at.h * a.os[2];
    store_row<kVec>(o, 1.0f / l_tot, op, a.d);
    // a row that saw nothing but masked keys: see canonical_bias
    if (g == 0)
        a.lse[(int64_t)at.bh * a.sq + i] = m == -kFltMax ? l_tot * kMaskedRowLse : m + logf(l_tot);
}

// dQ: dq_i = scale * sum_j ds_ij k_j,  ds = p (dp - delta),  dp = dO_i . v_j.  Also computes
// delta = rowsum(dO * O) of its rows and stores it for the dK / dV kernel, which runs second.
template <int DB, int kMode>
__global__ __launch_bounds__(kThreads, 2) void attn_f32_dq_kernel(const AttnArgs a_in) {
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    if (dropout) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    constexpr int kElems = Tile<DB, kVec>::kElems;
    float* ks = lds;
    float* vs = lds + 2 * kElems;
    const Place at(a, a.sq, true);
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const int wq0 = at.row0 + 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = wq0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];
    const float* gp = reinterpret_cast<const float*>(a.dout) + at.b * a.os[0] + at.h * a.os[2];
    const float* op = reinterpret_cast<const float*>(a.o) + at.b * a.os[0] + at.h * a.os[2];

    int j_lo, j_hi;
    key_range(a, at.row0, min(at.row0 + kRows, a.sq), j_lo, j_hi);
    j_hi = max(j_lo + 1, min(j_hi, has_bias ? padded_key_limit<kThreads, true>(a, at.b, at.h, lds) : a.sk));
    int t_lo = j_lo / kTile, t_hi = (j_hi + kTile - 1) / kTile;
    if (a.n_split > 1) split_tiles(a, at.split, t_lo, t_hi);

    Tile<DB, kVec> kt, vt;
    f32x4_t qf[DB], gf[DB], dq[DB];
    kt.load(kp, a.ks[1], t_lo * kTile, a.sk, a.d);
    vt.load(vp, a.vs[1], t_lo * kTile, a.sk, a.d);
    load_frags<kVec>(qf, qp, a.qs[1], i, a.sq, a.d, a.scale);
    load_frags<kVec>(gf, gp, a.os[1], i, a.sq, a.d, 1.0f);
    float delta = 0.f;
    {
        f32x4_t of[DB];
        load_frags<kVec>(of, op, a.os[1], i, a.sq, a.d, 1.0f);
#pragma unroll
        for (int x = 0; x < DB; ++x) {
            dq[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) delta = __builtin_fmaf(of[x][e], gf[x][e], delta);
        }
        delta = column_sum(delta);
    }
    const float lse_raw = i < a.sq ? a.lse[(int64_t)at.bh * a.sq + i] : 0.f;
    const float lse = lse_reference(lse_raw, 1.0f), inv_n = lse_row_factor(lse_raw);
    if (g == 0 && i < a.sq) a.delta[(int64_t)at.bh * a.sq + i] = delta;
    kt.store(ks, t_lo * kTile, a.sk, a.d);
    vt.store(vs, t_lo * kTile, a.sk, a.d);
    __syncthreads();

    const int wq_last = min(wq0 + 15, a.sq - 1);
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const float *kb = ks + slot * kElems, *vb = vs + slot * kElems;
        if (t + 1 < t_hi) {
            kt.load(kp, a.ks[1], (t + 1) * kTile, a.sk, a.d);
            vt.load(vp, a.vs[1], (t + 1) * kTile, a.sk, a.d);
        }
        const int j0 = t * kTile;
        const bool active = wq0 < a.sq && (!a.causal || j0 <= wq_last) &&
                            (a.window <= 0 || wq0 - (j0 + kTile - 1) < a.window);
        if (active) {
            const bool masked = j0 + kTile > a.sk || (a.causal && j0 + kTile - 1 > wq0) ||
                                (a.window > 0 && wq_last - j0 >= a.window);
            const Visible vis = keys_of_query(a, i, j0 + 4 * g, masked);
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                f32x4_t s = dot_rows<DB>(kb, 16 * h2, qf);
                f32x4_t dp = dot_rows<DB>(vb, 16 * h2, gf);
                uint32_t bits = 0xFu;
                if (dropout) bits = keep_keys(a, at.bh, i, j0 + 16 * h2 + 4 * g);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = j0 + 16 * h2 + 4 * g + r;
                    if (has_bias)
                        s[r] += bias_at(a, at.b, at.h, min(i, a.sq - 1), min(j, a.sk - 1));
                    if (dropout) dp[r] = (bits >> r) & 1u ? dp[r] * a.rng.inv_keep : 0.f;
                    const float ds = expf(s[r] - lse) * inv_n * (dp[r] - delta);
                    s[r] = vis(16 * h2 + r) ? ds : 0.f;
                }
                add_rows<DB>(kb, 16 * h2, s, dq);
            }
        }
        if (t + 1 < t_hi) {
            kt.store(ks + (slot ^ 1) * kElems, (t + 1) * kTile, a.sk, a.d);
            vt.store(vs + (slot ^ 1) * kElems, (t + 1) * kTile, a.sk, a.d);
        }
        __syncthreads();
    }
    if (i >= a.sq) return;
    if (a.n_split > 1) {
        store_row<kVec>(dq, a.scale, a.part + (at.part_row0 + i) * a.d, a.d);
        return;
    }
    float* dqp = reinterpret_cast<float*>(a.dq) + at.b * a.dqs[0] + (int64_t)i * a.dqs[1] +
                 at.h * a.dqs[2];
    store_row<kVec>(dq, a.scale, dqp, a.d);
}

// dK and dV: a wavefront owns 16 keys, queries stream through LDS.
//   dv_j = sum_i pdrop_ij dO_i          dk_j = scale * sum_i ds_ij q_i
template <int DB, int kMode>
__global__ __launch_bounds__(kThreads, 2) void attn_f32_dkv_kernel(const AttnArgs a_in) {
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    if (dropout) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    constexpr int kElems = Tile<DB, kVec>::kElems;
    float* qs = lds;
    float* gs = lds + 2 * kElems;
    float* rows = lds + 4 * kElems;  // [2][3][kTile]: lse reference, its factor, delta
    const Place at(a, a.sk, false);
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const int wk0 = at.row0 + 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = wk0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];
    const float* gp = reinterpret_cast<const float*>(a.dout) + at.b * a.os[0] + at.h * a.os[2];

    int i_lo, i_hi;
    query_range(a, at.row0, min(at.row0 + kRows, a.sk), i_lo, i_hi);
    // keys past the last unpadded one get no probability from any row
    if (at.row0 >= (has_bias ? padded_key_limit<kThreads, true>(a, at.b, at.h, lds) : a.sk)) i_hi = i_lo;
    int t_lo = i_lo / kTile, t_hi = (i_hi + kTile - 1) / kTile;
    if (a.n_split > 1) split_tiles(a, at.split, t_lo, t_hi);

    Tile<DB, kVec> qt, gt;
    f32x4_t kf[DB], vf[DB], dk[DB], dv[DB];
    float lse_r = 0.f, delta_r = 0.f;  // thread x < kTile: row x of the tile on its way
    auto request = [&](int t) __attribute__((always_inline)) {
        qt.load(qp, a.qs[1], t * kTile, a.sq, a.d);
        gt.load(gp, a.os[1], t * kTile, a.sq, a.d);
        if (threadIdx.x < kTile) {
            const int64_t row = (int64_t)at.bh * a.sq + min(t * kTile + (int)threadIdx.x, a.sq - 1);
            lse_r = a.lse[row];
            delta_r = a.delta[row];
        }
    };
    auto publish = [&](int t, int slot) __attribute__((always_inline)) {
        qt.store(qs + slot * kElems, t * kTile, a.sq, a.d);
        gt.store(gs + slot * kElems, t * kTile, a.sq, a.d);
        if (threadIdx.x < kTile) {
            float* r = rows + slot * 3 * kTile + threadIdx.x;
            r[0] = lse_reference(lse_r, 1.0f);
            r[kTile] = lse_row_factor(lse_r);
            r[2 * kTile] = delta_r;
        }
    };
    load_frags<kVec>(kf, kp, a.ks[1], j, a.sk, a.d, a.scale);
    load_frags<kVec>(vf, vp, a.vs[1], j, a.sk, a.d, 1.0f);
#pragma unroll
    for (int x = 0; x < DB; ++x) dk[x] = dv[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (t_lo < t_hi) {
        request(t_lo);
        publish(t_lo, 0);
    }
    __syncthreads();

    const int wk_last = min(wk0 + 15, a.sk - 1);
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const float *qb = qs + slot * kElems, *gb = gs + slot * kElems;
        const float* rb = rows + slot * 3 * kTile;
        if (t + 1 < t_hi) request(t + 1);
        const int i0 = t * kTile;
        const bool active = wk0 < a.sk && (!a.causal || i0 + kTile - 1 >= wk0) &&
                            (a.window <= 0 || i0 - wk_last < a.window);
        if (active) {
            const bool masked = i0 + kTile > a.sq || wk0 + 16 > a.sk ||
                                (a.causal && i0 < wk0 + 15) ||
                                (a.window > 0 && i0 + kTile - 1 - wk0 >= a.window);
            const Visible vis = queries_of_key(a, j, i0 + 4 * g, masked);
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                f32x4_t s = dot_rows<DB>(qb, 16 * h2, kf);
                f32x4_t dp = dot_rows<DB>(gb, 16 * h2, vf);
                const int r0 = 16 * h2 + 4 * g;
                const f32x4_t lse = *reinterpret_cast<const f32x4_t*>(rb + r0);
                const f32x4_t inv_n = *reinterpret_cast<const f32x4_t*>(rb + kTile + r0);
                const f32x4_t delta = *reinterpret_cast<const f32x4_t*>(rb + 2 * kTile + r0);
                uint32_t bits = 0xFu;
                if (dropout) bits = keep_queries(a, at.bh, i0 + r0, wk0);
                f32x4_t pd;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = i0 + r0 + r;
                    if (has_bias)
                        s[r] += bias_at(a, at.b, at.h, min(i, a.sq - 1), min(j, a.sk - 1));
                    const float p = expf(s[r] - lse[r]) * inv_n[r];
                    const float keep = dropout ? ((bits >> r) & 1u ? a.rng.inv_keep : 0.f) : 1.f;
                    const bool seen = vis(16 * h2 + r);
                    pd[r] = seen ? p * keep : 0.f;
                    s[r] = seen ? p * (dp[r] * keep - delta[r]) : 0.f;
                }
                add_rows<DB>(gb, 16 * h2, pd, dv);
                add_rows<DB>(qb, 16 * h2, s, dk);
            }
        }
        if (t + 1 < t_hi) publish(t + 1, slot ^ 1);
        __syncthreads();
    }
    if (j >= a.sk) return;
    if (a.n_split > 1) {
        float* part = a.part + (at.part_row0 + j) * a.d;
        store_row<kVec>(dk, a.scale, part, a.d);
        store_row<kVec>(dv, 1.0f,
                        part + (int64_t)a.n_split * a.batch * a.heads * a.sk * a.d, a.d);
        return;
    }
    float* dkp = reinterpret_cast<float*>(a.dk) + at.b * a.dks[0] + (int64_t)j * a.dks[1] +
                 at.h * a.dks[2];
    float* dvp = reinterpret_cast<float*>(a.dv) + at.b * a.dvs[0] + (int64_t)j * a.dvs[1] +
                 at.h * a.dvs[2];
    store_row<kVec>(dk, a.scale, dkp, a.d);
    store_row<kVec>(dv, 1.0f, dvp, a.d);
}

enum class Which { kFwd, kDq, kDkv };

// DB = 16-wide blocks of the head dimension
template <int DB, Which kWhich, int kMode, int kHalves = 1>
int launch(const AttnArgs& a, hipStream_t st) {
    const int n_rows = kWhich == Which::kDkv ? a.sk : a.sq;
    const int64_t blocks =
        (int64_t)((n_rows + kRows - 1) / kRows) * a.batch * a.heads * a.n_split;
    if (blocks <= 0 || blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    if constexpr (kWhich == Which::kFwd && kHalves == 1) {
        if (blocks <= kHalvesBlocks) return launch<DB, kWhich, kMode, 2>(a, st);
    }
    const size_t smem = (4 * kHalves * kTile * kPitchOf<DB> +
                         (kWhich == Which::kDkv ? 6 * kTile : 0)) *
                        sizeof(float);
    auto kern = kWhich == Which::kFwd  ? attn_f32_fwd_kernel<DB, kMode, kHalves>
                : kWhich == Which::kDq ? attn_f32_dq_kernel<DB, kMode>
                                       : attn_f32_dkv_kernel<DB, kMode>;
    static std::atomic<uint64_t> lds_ready{0};
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_ready) != SLAPO_OK)
        return SLAPO_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kHalves * kThreads), smem, st, a);
    return check_launch();
}

template <Which kWhich, int DB>
int dispatch_mode(const AttnArgs& a, hipStream_t st) {
    uintptr_t odd = (uintptr_t)(a.d & 3);
    auto rows = [&](const void* p, const int64_t (&s)[3]) {
        odd |= (reinterpret_cast<uintptr_t>(p) & 15) | (uintptr_t)((s[0] | s[1] | s[2]) & 3);
    };
    rows(a.q, a.qs), rows(a.k, a.ks), rows(a.v, a.vs), rows(a.o, a.os);
    if (kWhich != Which::kFwd) rows(a.dout, a.os);
    if (kWhich == Which::kDq) rows(a.dq, a.dqs);
    if (kWhich == Which::kDkv) rows(a.dk, a.dks), rows(a.dv, a.dvs);
    if (odd) return launch<DB, kWhich, kGeneral>(a, st);
    if (a.dropout)
        return a.has_bias ? launch<DB, kWhich, 3>(a, st) : launch<DB, kWhich, 2>(a, st);
    return a.has_bias ? launch<DB, kWhich, 1>(a, st) : launch<DB, kWhich, 0>(a, st);
}

template <Which kWhich>
int dispatch(const AttnArgs& a, hipStream_t st) {
    switch ((a.d + 15) / 16) {
        case 1:
        case 2: return dispatch_mode<kWhich, 2>(a, st);
        case 3:
        case 4: return dispatch_mode<kWhich, 4>(a, st);
        case 5: return dispatch_mode<kWhich, 5>(a, st);
        case 6: return dispatch_mode<kWhich, 6>(a, st);
        case 7:
        case 8: return dispatch_mode<kWhich, 8>(a, st);
        default: return SLAPO_ERR_SHAPE;
    }
}

}  // namespace

namespace slapo {

int attn_fwd_f32(const AttnArgs& a, hipStream_t st) { return dispatch<Which::kFwd>(a, st); }
int attn_bwd_dq_f32(const AttnArgs& a, hipStream_t st) { return dispatch<Which::kDq>(a, st); }
int attn_bwd_f32(const AttnArgs& a, hipStream_t st) { return dispatch<Which::kDkv>(a, st); }

}  // namespace slapo
