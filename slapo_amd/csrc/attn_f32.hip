// Attention forward and backward for fp32 tensors, the kernels behind dtype == SLAPO_F32, whose
// parity bar is 1e-5 absolute.
//
// Products run on the bf16 matrix instructions without giving up fp32: an operand is the sum of three
// bf16 numbers, x = h + m + l (h = bf16(x), m = bf16(x - h), l = bf16(x - h - m): 8 + 8 + 8 mantissa
// bits), and x y = hh + (hm + mh) + (mm + hl + lh) + O(2^-25 |x y|), six v_mfma_f32_16x16x32_bf16 with
// exact products and fp32 sums.  The parts have the three ranges that fp32's has not:
//  * l's last bit is 2^-24 x: below 2^-102 it leaves bf16's normal numbers.  V, K, Q, dO, the
//    probabilities and dS are therefore split at 2^24 times their size (kUp), exactly, and the results
//    are lowered again: every normal fp32 number is the exact sum of its parts.  Only scores need no such
//    care: what their operands lose is at most 2^-125 each, 2^-58 of a score beside numbers below 2^60.
//  * What bf16 rounds to infinity, and infinities, have no finite parts.  A workgroup that meets a
//    magnitude above 2^36 (2^60 at the size held: kTop), or whose results are not all finite, writes
//    nothing and runs its rows again on v_mfma_f32_16x16x4_f32 (Full8), whose products are fp32's own:
//    infinity times infinity is one.  Where all do, a call takes 2.4 times as long (forward and
//    backward of B4 S512 H16 D64 133 -> 317 us).
//  * Probabilities below 2^-126 are zero in the first pass (v_exp_f32).
//
// v_mfma_f32_16x16x32_bf16 (one wavefront, lane l, i = l % 16, g = l / 16):
//   A operand: lane holds A[row i][k-slots 8 g .. 8 g + 7];   B operand: the same slots of column i;
//   C/D:       register r of lane l is element (row 4 g + r, column i).
// The k-slots may stand for any data as long as A and B agree, and so may the rows of A:
//  * products over the head dimension (S = QK^T, dP = dO V^T): slot 8 g + e of step t is element
//    32 t + 8 g + e, a 16-byte read per plane; MFMA row 4 g + r is tile row 4 r + lane_row(g) of a
//    group of 16 (lane_row swaps the two bits of g);
//  * products over keys or queries (PV, dS K, P^T dO, dS^T Q): the accumulator registers r of two
//    such groups are slots r and 4 + r, so probabilities never leave registers, and the other
//    operand comes from the row-major tile by two transposing reads per plane.
// With that row order and a pitch of an odd number of 16-byte units both kinds of read touch every
// bank once.
//
// A workgroup owns 16 rows per wavefront (queries in forward and dQ, keys in dK/dV); the other side
// streams through LDS in tiles of 32 rows, double buffered, staged through registers and split into its
// planes on the way.  Per 16 x 32 scores and wavefront (forward, head_dim 64) that is 768 matrix
// cycles -- the fp32 matrix instructions take 2048 --, about 200 vector instructions (half of them
// the splitting of the tile and of the probabilities) and 24 KB of LDS reads: no one of the three
// binds, their sum does.  fp32 matrix instructions in the same layout -> these: forward B4 S512
// H16 D64 50.9 -> 33.1 us (83 -> 130 TFLOP/s), B16 S512 H16 D64 184 -> 102, B2 S2048 H16 D128 701 -> 357
// (193 TFLOP/s; the fp32 instructions stop at 157, six bf16 products for one at about 222); forward and
// backward B4 S512 H16 D64 210 -> 124, B4 S1024 H8 D80 554 -> 334, B1 S1024 H8 D128 causal 233 -> 146.
// Errors against 64 bits (2-norm) at B4 S512 H16 D64: output 4.1e-7 -> 2.0e-7, gradients 6.2e-7 ->
// 4.3e-7; at B2 S2048 H16 D128 output 9.3e-7 -> 3.7e-7.
// What the sizes held above (kUp) and the largest magnitude cost: B4 S512 H16 D64 32.7 -> 33.1 us
// forward, 150.0 -> 152.5 with a padding mask and backward; what it gave, by fewer branches: B4 S700 H12
// D80 causal and padded 67.9 -> 66.0 forward, B2 S1000 H6 D96 window 200 85.8 -> 82.3 with backward.
//
// Reference semantics: slapo/op/attention.py:163-181 (attention_bmk) and its autograd.
#include <type_traits>

#include "attn_common.h"

using namespace slapo;

namespace {

constexpr int kTile = 32;  // streamed rows per LDS tile
// Wavefronts per workgroup (16 rows each).  Eight split a tile once for 128 rows where four do it for
// 64, and let head_dim 128, whose 104 KB of tiles leave a CU one workgroup, have two wavefronts per
// SIMD (B1 S1024 H8 D128 causal, forward and backward: 146 against 198 us).  At head_dim 65-96
// two workgroups of four fit a CU and balance causal and windowed calls better (B2 S1000 H6 D96
// window 200: 87 against 127 us; without a mask equal).  Up to 64 it takes workgroups enough:
constexpr int64_t kWideBwd = 512;   // in units of 64 rows: B4 S512 H16 D64 (512) 125 against 132 us
                                    // forward and backward, B2 S777 H12 D64 (312) padded, p 0.1 305
                                    // against 283; a forward gains at once (288: 32.8 against 34.8)
// Small forward calls up to head_dim 96 run kHalves = 2: eight wavefronts, two per 16 query rows, each
// with one half of a tile of 64 keys and a softmax state of its own, merged at the end through LDS (B1
// S256 H8 D64, 32 units: 12.3 us against 15.6 with four wavefronts and 18.1 with eight times 16 rows;
// B4 S292 H4 D72, 80 units: 19.2 against 25.7; B2 S512 H8 D72, 128 units: 32.2 against 27.6).
constexpr int64_t kHalvesBelow = 128;
// LDS and registers leave a SIMD four of a forward's wavefronts up to head_dim 64, else two.
constexpr int per_simd(int db, int waves) { return db <= 4 && waves >= 8 ? 4 : 2; }
// ... of a backward kernel's four up to head_dim 32 where no dropout is drawn for columns, else two.
constexpr int per_simd_bwd(int db, bool draws) { return db <= 2 && !draws ? 4 : 2; }
// The forward moves its softmax reference when a score stands more than this above it, in log2 units.
constexpr float kPartsAhead = 8.0f;

typedef Mma<bf16_t>::frag frag_t;
__device__ __forceinline__ f32x4_t splat(float v) { return f32x4_t{v, v, v, v}; }
// The two forms of eight fp32 numbers: their bf16 parts, and themselves.
struct Split8 {
    u32x4_t h, m, l;
};
struct Full8 {
    f32x4_t a, b;
};
// (see read_again)
template <bool kParts>
__device__ __forceinline__ int thread_of() {
    int t = threadIdx.x;
    if constexpr (!kParts) asm("" : "+v"(t));
    return t;
}
template <bool kParts>
using operand_t = std::conditional_t<kParts, Split8, Full8>;
__device__ __forceinline__ frag_t frag(u32x4_t v) { return __builtin_bit_cast(frag_t, v); }
// c (and, in `small`, the five smaller products) += A B of fp32 operands
__device__ __forceinline__ void mma(const Split8& a, const Split8& b, f32x4_t& c, f32x4_t& small) {
    small = Mma<bf16_t>::mma16(frag(a.l), frag(b.h), small);
    small = Mma<bf16_t>::mma16(frag(a.h), frag(b.l), small);
    small = Mma<bf16_t>::mma16(frag(a.m), frag(b.m), small);
    small = Mma<bf16_t>::mma16(frag(a.m), frag(b.h), small);
    small = Mma<bf16_t>::mma16(frag(a.h), frag(b.m), small);
    c = Mma<bf16_t>::mma16(frag(a.h), frag(b.h), c);
}
// c += A B over four k-slots, slot g of this lane's column
__device__ __forceinline__ void mma4(float a, float b, f32x4_t& c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float low_half(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float high_half(uint32_t v) {
    return __builtin_bit_cast(float, v & 0xFFFF0000u);
}
__device__ __forceinline__ void split2(float x, float y, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack2<bf16_t>(x, y);
    x -= low_half(h), y -= high_half(h);
    m = pack2<bf16_t>(x, y);
    l = pack2<bf16_t>(x - low_half(m), y - high_half(m));
}
template <bool kParts>
__device__ __forceinline__ operand_t<kParts> operand(const f32x4_t& a, const f32x4_t& b) {
    if constexpr (kParts) {
        uint32_t h[4], m[4], l[4];
        split2(a[0], a[1], h[0], m[0], l[0]);
        split2(a[2], a[3], h[1], m[1], l[1]);
        split2(b[0], b[1], h[2], m[2], l[2]);
        split2(b[2], b[3], h[3], m[3], l[3]);
        return {u32x4_t{h[0], h[1], h[2], h[3]}, u32x4_t{m[0], m[1], m[2], m[3]},
                u32x4_t{l[0], l[1], l[2], l[3]}};
    } else {
        return {a, b};
    }
}
// In parts everything but the scores' own operands is held kUp times its size: the last part of a number of
// 2^-126 is then one of 2^-126, where bf16 has all its bits, instead of one of 2^-150, where it has none.
constexpr float kUp = 0x1p24f;
template <bool kParts>
constexpr float lift = kParts ? kUp : 1.0f;
// What a pass in bf16 parts may see, at the size held: up to it every part, every score and every dO v is
// finite, and a result that went wrong on the way (a sum past fp32's range) is not.
constexpr float kTop = 0x1p60f;
// top = the largest magnitude so far (not of NaN, which reaches the results)
__device__ __forceinline__ void track(float& top, const f32x4_t& v) {
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(v[0]), "v"(v[1]));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(v[2]), "v"(v[3]));
}
// 0, or NaN once a result is not finite
template <int DB>
__device__ __forceinline__ float not_finite(const f32x4_t (&acc)[DB], float so_far = 0.f) {
#pragma unroll
    for (int x = 0; x < DB; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) so_far = __builtin_fmaf(acc[x][e], 0.f, so_far);
    return so_far;
}
// 2^x: of parts, zero below 2^-126
template <bool kParts>
__device__ __forceinline__ float exp2_of(float x) {
    return kParts ? fast_exp2(x) : __builtin_exp2f(x);
}
// Whether `ok` holds in every thread of the workgroup's kWaves wavefronts; `votes` is theirs alone.
template <int kWaves>
__device__ __forceinline__ bool everywhere(bool ok, int* votes) {
    const bool wave_ok = __builtin_amdgcn_ballot_w64(!ok) == 0;
    if ((threadIdx.x & 63) == 0) votes[threadIdx.x >> 6] = wave_ok;
    __syncthreads();
    int all = 1;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) all &= votes[w];
    return __builtin_amdgcn_readfirstlane(all) != 0;
}
// Tile row (of a group of 16) of accumulator register r of lane-group g: 4 r + lane_row(g).
__device__ __forceinline__ int lane_row(int g) { return (g & 1) * 2 + (g >> 1); }
// Across the four lanes that share a column (l, l ^ 16, l ^ 32, l ^ 48)
__device__ __forceinline__ void swap16(float v, float& even, float& odd) {
    float a = v, b = v;  // the odd rows of 16 lanes of one against the even rows of the other
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    even = a, odd = b;
}
__device__ __forceinline__ float column_max(float v) {
    float a, b;
    swap16(v, a, b);
    return max_xor32(fmaxf(a, b));
}
__device__ __forceinline__ float column_sum(float v) {
    float a, b;
    swap16(v, a, b);
    return sum_xor32(a + b);
}

__device__ __forceinline__ float bias_at(const AttnArgs& a, int b, int h, int i, int j) {
    return bias_log2(bias_load(
        a, b * a.bs[0] + h * a.bs[1] + (int64_t)i * a.bs[2] + (int64_t)j * a.bs[3]));
}

// Steps of 32 over the head dimension, and the LDS row pitch of a tile's plane in elements
template <int DB>
constexpr int kStepsOf = (DB + 1) / 2;
template <int DB>
constexpr int kPitchOf = 32 * kStepsOf<DB> + 8;
template <int DB>
constexpr int kFullPitchOf = 32 * kStepsOf<DB> + 4;  // of a tile of fp32 numbers, in floats

// Builds of each kernel: kMode & 1 = with a bias, kMode & 2 = with dropout, for tensors whose rows are
// 16-byte aligned with d % 4 == 0; kGeneral serves every other layout element by element and decides
// about bias and dropout when it runs.
constexpr int kGeneral = 4;

// A tile of kTileRows rows on its way from global memory to LDS, where it stands as three bf16 planes or,
// in less of the same place, as it is.  Rows past the end are clamped, columns past d read as zero.
template <int DB, bool kVec, int kTileRows, int kBlock, bool kParts>
struct Tile {
    static constexpr int kPitch = kPitchOf<DB>;
    static constexpr int kPlane = kTileRows * kPitch;
    static constexpr int kElems = 3 * kPlane;
    static_assert(sizeof(float) * kFullPitchOf<DB> <= 3 * sizeof(bf16_t) * kPitch);
    static constexpr int kPerRow = 8 * kStepsOf<DB>;
    static constexpr int kChunks = kTileRows * kPerRow;
    static constexpr int kPer = (kChunks + kBlock - 1) / kBlock;
    f32x4_t r[kPer];

    __device__ __forceinline__ void load(const float* base, int64_t stride, int row0, int n_rows,
                                         int d) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = thread_of<kParts>() + u * kBlock;
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
    // times kUp where kLift; `top` tracked where kScores (an operand of the scores)
    template <bool kLift, bool kScores>
    __device__ __forceinline__ void store(bf16_t* lds, int row0, int n_rows, int d, float& top) {
        if (row0 + kTileRows > n_rows || d < 32 * kStepsOf<DB>) {  // uniform
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int c = thread_of<kParts>() + u * kBlock;
                const int row = c / kPerRow, col = 4 * (c % kPerRow);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row0 + row >= n_rows || col + e >= d) r[u][e] = 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int c = thread_of<kParts>() + u * kBlock;
            if (kChunks % kBlock != 0 && c >= kChunks) continue;
            const int row = c / kPerRow, col = 4 * (c % kPerRow);
            if constexpr (kParts) {
                uint32_t h[2], m[2], l[2];
                if (kLift) r[u] *= kUp;
                if (kScores) track(top, r[u]);
                split2(r[u][0], r[u][1], h[0], m[0], l[0]);
                split2(r[u][2], r[u][3], h[1], m[1], l[1]);
                bf16_t* p = lds + row * kPitch + col;
                *reinterpret_cast<u32x2_t*>(p) = u32x2_t{h[0], h[1]};
                *reinterpret_cast<u32x2_t*>(p + kPlane) = u32x2_t{m[0], m[1]};
                *reinterpret_cast<u32x2_t*>(p + 2 * kPlane) = u32x2_t{l[0], l[1]};
            } else {
                float* p = reinterpret_cast<float*>(lds) + row * kFullPitchOf<DB> + col;
                *reinterpret_cast<f32x4_t*>(p) = r[u];
            }
        }
    }
};

// Row `row` of a tensor as this lane holds it: elements 32 t + 8 g .. + 7 in f[2 t], f[2 t + 1].
template <bool kParts, bool kVec, int KS>
__device__ __forceinline__ void load_row(f32x4_t (&f)[2 * KS], const float* base, int64_t stride,
                                         int row, int n_rows, int d, float scale) {
    const int g = (thread_of<kParts>() & 63) >> 4;
    const float* p = base + (int64_t)min(row, n_rows - 1) * stride;
#pragma unroll
    for (int t = 0; t < 2 * KS; ++t) {
        const int col = 32 * (t >> 1) + 8 * g + 4 * (t & 1);
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
template <bool kParts, int KS>
__device__ __forceinline__ void hold_row(operand_t<kParts> (&f)[KS], const f32x4_t (&v)[2 * KS]) {
#pragma unroll
    for (int t = 0; t < KS; ++t) f[t] = operand<kParts>(v[2 * t], v[2 * t + 1]);
}
template <int N>
__device__ __forceinline__ void track_row(float& top, const f32x4_t (&v)[N]) {
#pragma unroll
    for (int t = 0; t < N; ++t) track(top, v[t]);
}

// small + A B over the head dimension: A = 16 tile rows from row `r0` on, B = this lane's fragments.
template <int DB, int kPlane>
__device__ __forceinline__ f32x4_t dot_rows(const bf16_t* tile, int r0,
                                            const Split8 (&f)[kStepsOf<DB>],
                                            f32x4_t small = f32x4_t{0.f, 0.f, 0.f, 0.f}) {
    const int lane = thread_of<true>() & 63, i = lane & 15;
    const bf16_t* p = tile + (r0 + 4 * (i & 3) + lane_row(i >> 2)) * kPitchOf<DB> + 8 * (lane >> 4);
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kStepsOf<DB>; ++t) {
        const bf16_t* q = p + 32 * t;
        const Split8 v = {*reinterpret_cast<const u32x4_t*>(q),
                          *reinterpret_cast<const u32x4_t*>(q + kPlane),
                          *reinterpret_cast<const u32x4_t*>(q + 2 * kPlane)};
        mma(v, f[t], c, small);
    }
    return c + small;
}
template <int DB, int kPlane>
__device__ __forceinline__ f32x4_t dot_rows(const bf16_t* tile, int r0,
                                            const Full8 (&f)[kStepsOf<DB>],
                                            f32x4_t small = f32x4_t{0.f, 0.f, 0.f, 0.f}) {
    const int lane = thread_of<false>() & 63, i = lane & 15;
    const float* p = reinterpret_cast<const float*>(tile) +
                     (r0 + 4 * (i & 3) + lane_row(i >> 2)) * kFullPitchOf<DB> + 8 * (lane >> 4);
    f32x4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < kStepsOf<DB>; ++t) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p + 32 * t);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(p + 32 * t + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) mma4(a[e], f[t].a[e], c);
#pragma unroll
        for (int e = 0; e < 4; ++e) mma4(b[e], f[t].b[e], c);
    }
    return c + small;
}
// acc[x] += A B over the 32 tile rows: A = columns 16 x .. 16 x + 15 of those rows (transposed), B =
// w, slots r and 4 + r of it being rows 4 r + lane_row(g) and 16 more of this lane's column.
template <int DB, int kPlane>
__device__ __forceinline__ void add_rows(const bf16_t* tile, const Split8& w, f32x4_t (&acc)[DB],
                                         f32x4_t (&small)[DB]) {
    const int lane = thread_of<true>() & 63;
    const bf16_t* p = tile +
                      (4 * ((lane & 15) >> 2) + lane_row(lane >> 4)) * kPitchOf<DB> + 4 * (lane & 3);
    auto columns = [&](const bf16_t* q) __attribute__((always_inline)) {
        const u32x2_t a = lds_read_tr16(q), b = lds_read_tr16(q + 16 * kPitchOf<DB>);
        return u32x4_t{a.x, a.y, b.x, b.y};
    };
#pragma unroll
    for (int x = 0; x < DB; ++x) {
        const bf16_t* q = p + 16 * x;
        const Split8 v = {columns(q), columns(q + kPlane), columns(q + 2 * kPlane)};
        mma(v, w, acc[x], small[x]);
    }
}

template <int DB, int kPlane>
__device__ __forceinline__ void add_rows(const bf16_t* tile, const Full8& w, f32x4_t (&acc)[DB],
                                         f32x4_t (&)[DB]) {
    const int lane = thread_of<false>() & 63;
    const float* p = reinterpret_cast<const float*>(tile) +
                     lane_row(lane >> 4) * kFullPitchOf<DB> + (lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r, p += 4 * kFullPitchOf<DB>)
#pragma unroll
        for (int x = 0; x < DB; ++x) {
            mma4(p[16 * x], w.a[r], acc[x]);
            mma4(p[16 * kFullPitchOf<DB> + 16 * x], w.b[r], acc[x]);
        }
}

// Writes this lane's column of acc (element 16 x + 4 g + r in acc[x][r]), lowered by `down` (a power of
// two, so that mul meets what fp32 sums would be), times mul as row `row`.
template <bool kParts, bool kVec, int DB>
__device__ __forceinline__ void store_row(const f32x4_t (&acc)[DB], float down, float mul,
                                          float* row, int d) {
    const int g = (thread_of<kParts>() & 63) >> 4;
#pragma unroll
    for (int x = 0; x < DB; ++x) {
        const int col = 16 * x + 4 * g;
        if constexpr (kVec) {
            if (col < d) *reinterpret_cast<f32x4_t*>(row + col) = acc[x] * down * mul;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < d) row[col + e] = acc[x][e] * down * mul;
        }
    }
}

// Keep bits (bit r: key j + r) of query i and the kKeys keys from j on, j % 4 == 0.
template <int kKeys>
__device__ __forceinline__ uint32_t keep_keys(const AttnArgs& a, int bh, int i, int j) {
    const uint64_t e = ((uint64_t)bh * a.sq + (uint64_t)i) * (uint64_t)a.sk + (uint64_t)j;
    if (i >= a.sq || j >= a.sk) return 0;
    if (a.dropout != 1) return dropout_keep_run<kKeys>(a.rng, e);
    uint32_t bits = dropout_keep4_pow2(a.rng, e >> 2);
#pragma unroll
    for (int k = 4; k < kKeys; k += 4)
        if (j + k < a.sk) bits |= dropout_keep4_pow2(a.rng, (e + (uint64_t)k) >> 2) << k;
    return bits;
}
// Keep bits of query i (the lane's column) and the 32 keys from j0 on: a Philox block covers four
// consecutive keys, so each of the four lanes of a query draws eight keys and they exchange them.
template <bool kParts>
__device__ __forceinline__ uint32_t keep_keys32(const AttnArgs& a, int bh, int i, int j0) {
    const int at = 8 * ((thread_of<kParts>() & 63) >> 4);
    uint32_t bits = keep_keys<8>(a, bh, i, j0 + at) << at;
    bits |= (uint32_t)__shfl_xor((int)bits, 16, 64);
    return bits | (uint32_t)__shfl_xor((int)bits, 32, 64);
}
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xF, 0xF, false);
}
// The same for a lane whose registers are the queries i + 4 r and whose key is j0 + l % 16 (bit r:
// query i + 4 r): a Philox block covers four consecutive keys, i.e. the four lanes of a quad, so
// lane c of a quad draws the block of query i + 4 c and the quad exchanges them.
template <bool kParts>
__device__ __forceinline__ uint32_t keep_queries(const AttnArgs& a, int bh, int i, int j0) {
    const int c = thread_of<kParts>() & 3, j = j0 + (thread_of<kParts>() & 15);
    const uint32_t mine = keep_keys<4>(a, bh, i + 4 * c, j - c);
    return ((dpp<0x00>(mine) >> c) & 1u) | (((dpp<0x55>(mine) >> c) & 1u) << 1) |
           (((dpp<0xAA>(mine) >> c) & 1u) << 2) | (((dpp<0xFF>(mine) >> c) & 1u) << 3);
}

// What a workgroup of the query-owning kernels works on: heaviest query tiles first, the heads as
// the fast index so that the tiles of one head share an XCD's L2.
struct Place {
    int b, h, bh, row0, split;
    int64_t part_row0;  // of the split's partial result, rows of all (batch, head) pairs
    // kRows rows per workgroup
    __device__ __forceinline__ Place(const AttnArgs& a, int n_rows, int kRows, bool last_first) {
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

// The kernel's arguments once more, for the pass on fp32 instructions (thread_of: likewise).  What the
// compiler knows to be the same it would compute once and hold in registers through the first pass,
// which has none left for a pass that hardly ever follows.
__device__ __forceinline__ AttnArgs read_again() {
    typedef const __attribute__((address_space(4))) uint32_t* words_t;
    words_t p = (words_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    uint32_t w[sizeof(AttnArgs) / sizeof(uint32_t)];
    static_assert(sizeof(AttnArgs) % sizeof(uint32_t) == 0);
#pragma unroll
    for (unsigned i = 0; i < sizeof(w) / sizeof(w[0]); ++i) w[i] = p[i];
    AttnArgs a;
    __builtin_memcpy(&a, w, sizeof(a));
    if (a.dropout) resolve_device_state(a.rng);
    return a;
}

// Which elements c of a lane's run are visible: lo <= c <= hi.
struct Visible {
    int lo, hi;
    __device__ __forceinline__ bool operator()(int c) const { return c >= lo && c <= hi; }
};
// the run starts at key `first` of query i
__device__ __forceinline__ Visible keys_of_query(const AttnArgs& a, int i, int first) {
    return {(a.window > 0 ? i - a.window + 1 : 0) - first,
            (a.causal ? min(i, a.sk - 1) : a.sk - 1) - first};
}
// the run starts at query `first` of key j
__device__ __forceinline__ Visible queries_of_key(const AttnArgs& a, int j, int first) {
    return {(a.causal ? j : 0) - first,
            (a.window > 0 ? min(j + a.window, a.sq) - 1 : a.sq - 1) - first};
}

// One pass of a workgroup over its rows, tiles t_lo .. t_hi - 1.  false (of kParts alone): nothing is
// written, the caller has the other form do it.
template <int DB, int kMode, int kWaves, int kHalves, bool kParts>
__device__ __forceinline__ bool fwd_pass(const AttnArgs& a, const Place& at, int t_lo, int t_hi,
                                         float* lds) {
    constexpr int kFwdThreads = kHalves * kWaves * 64, kFwdTile = kHalves * kTile;
    constexpr int KS = kStepsOf<DB>;
    constexpr bool kVec = kMode != kGeneral;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    constexpr float kAhead = kParts ? kPartsAhead : 0.f, kLift = lift<kParts>;
    typedef Tile<DB, kVec, kFwdTile, kFwdThreads, kParts> tile_t;
    constexpr int kElems = tile_t::kElems, kPlane = tile_t::kPlane;
    bf16_t* ks = reinterpret_cast<bf16_t*>(lds);  // K[2][tile]
    bf16_t* vs = ks + 2 * kElems;                 // V[2][tile]
    const int lane = thread_of<kParts>() & 63, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(thread_of<kParts>() >> 6);
    const int wq0 = at.row0 + 16 * (wave % kWaves);
    const int half = wave / kWaves;  // of every tile's keys
    const int row_g = lane_row(g);
    const int i = wq0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];

    float top = 0.f;
    tile_t kt, vt;
    operand_t<kParts> qf[KS];
    f32x4_t o[DB], o_small[DB];  // (mma)
    kt.load(kp, a.ks[1], t_lo * kFwdTile, a.sk, a.d);
    vt.load(vp, a.vs[1], t_lo * kFwdTile, a.sk, a.d);
    {
        f32x4_t q[2 * KS];
        load_row<kParts, kVec, KS>(q, qp, a.qs[1], i, a.sq, a.d, a.scale_log2);
        if (kParts) track_row(top, q);
        hold_row<kParts, KS>(qf, q);
    }
#pragma unroll
    for (int x = 0; x < DB; ++x) o[x] = o_small[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;  // m: in log2 units, as the scores are; l: this lane's share of the row sum
    kt.template store<false, true>(ks, t_lo * kFwdTile, a.sk, a.d, top);
    vt.template store<kParts, true>(vs, t_lo * kFwdTile, a.sk, a.d, top);
    __syncthreads();

    const int wq_last = min(wq0 + 15, a.sq - 1);
    const float kept = dropout ? a.rng.inv_keep * kLift : kLift;
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const int part = half * kTile * (kParts ? tile_t::kPitch : 2 * kFullPitchOf<DB>);
        const bf16_t *kb = ks + slot * kElems + part, *vb = vs + slot * kElems + part;
        if (kParts && t + 1 < t_hi) {
            kt.load(kp, a.ks[1], (t + 1) * kFwdTile, a.sk, a.d);
            vt.load(vp, a.vs[1], (t + 1) * kFwdTile, a.sk, a.d);
        }
        const int j0 = t * kFwdTile + half * kTile;
        const bool active = wq0 < a.sq && j0 < a.sk && (!a.causal || j0 <= wq_last) &&
                            (a.window <= 0 || wq0 - (j0 + kTile - 1) < a.window);
        if (active) {  // uniform per wavefront
            f32x4_t s[2];
            s[0] = dot_rows<DB, kPlane>(kb, 0, qf);
            s[1] = dot_rows<DB, kPlane>(kb, 16, qf);
            const bool masked = j0 + kTile > a.sk || (a.causal && j0 + kTile - 1 > wq0) ||
                                (a.window > 0 && wq_last - j0 >= a.window);
            if (has_bias) {
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        s[h2][r] += bias_at(a, at.b, at.h, min(i, a.sq - 1),
                                            min(j0 + 16 * h2 + 4 * r + row_g, a.sk - 1));
            }
            if (masked) {  // uniform
                const Visible vis = keys_of_query(a, i, j0 + row_g);
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!vis(16 * h2 + 4 * r)) s[h2][r] = -INFINITY;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, fmaxf(s[0][r], s[1][r]));
            mx = column_max(mx);
            // moved lazily: probabilities stay at or below 2^kAhead
            const bool move = mx - m > kAhead;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(move) != 0, 0)) {
                const float m_new = move ? mx : m;
                const float alpha = m == -INFINITY ? 0.f : exp2_of<kParts>(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int x = 0; x < DB; ++x) o[x] *= alpha, o_small[x] *= alpha;
            }
            const float m_ref = m == -INFINITY ? 0.f : m;
            uint32_t bits = 0u;
            if (dropout) bits = keep_keys32<kParts>(a, at.bh, i, j0) >> row_g;
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float p = exp2_of<kParts>(s[h2][r] - m_ref);
                    l += p;
                    const bool drop = dropout && ((bits >> (16 * h2 + 4 * r)) & 1u) == 0;
                    s[h2][r] = drop ? 0.f : p * kept;
                }
            add_rows<DB, kPlane>(vb, operand<kParts>(s[0], s[1]), o, o_small);
        }
        if (t + 1 < t_hi) {
            if (!kParts) kt.load(kp, a.ks[1], (t + 1) * kFwdTile, a.sk, a.d);
            kt.template store<false, true>(ks + (slot ^ 1) * kElems, (t + 1) * kFwdTile, a.sk, a.d, top);
            if (!kParts) vt.load(vp, a.vs[1], (t + 1) * kFwdTile, a.sk, a.d);
            vt.template store<kParts, true>(vs + (slot ^ 1) * kElems, (t + 1) * kFwdTile, a.sk, a.d, top);
        }
        __syncthreads();
    }
    float l_tot = column_sum(l);
#pragma unroll
    for (int x = 0; x < DB; ++x) o[x] += o_small[x];
    if constexpr (kParts) {  // (the votes lie behind the halves' states)
        const bool ok = top <= kTop && not_finite(o) == 0.f;
        int* votes = reinterpret_cast<int*>(ks + 4 * kElems) - kHalves * kWaves;
        if (!everywhere<kHalves * kWaves>(ok, votes)) return false;
    }
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
        if (half != 0) return true;
        const float m2 = state[4 * DB * 64], m_all = fmaxf(m, m2);
        const float w1 = m == -INFINITY ? 0.f : exp2_of<kParts>(m - m_all);
        const float w2 = m2 == -INFINITY ? 0.f : exp2_of<kParts>(m2 - m_all);
        l_tot = l_tot * w1 + state[(4 * DB + 1) * 64] * w2;
        m = m_all;
#pragma unroll
        for (int x = 0; x < DB; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[x][e] = o[x][e] * w1 + state[(4 * x + e) * 64] * w2;
    }
    if (i >= a.sq) return true;
    if (a.n_split > 1) {
        store_row<kParts, kVec>(o, 1.0f / (kLift * kLift), 1.0f, a.part + (at.part_row0 + i) * a.d, a.d);
        if (g == 0) {
            float* ml = a.part + (int64_t)a.n_split * a.batch * a.heads * a.sq * a.d +
                        2 * (at.part_row0 + i);
            ml[0] = m, ml[1] = l_tot;
        }
        return true;
    }
    float* op = reinterpret_cast<float*>(a.o) + at.b * a.os[0] + (int64_t)i * a.os[1] +
                at.h * a.os[2];
    store_row<kParts, kVec>(o, 1.0f / (kLift * kLift), 1.0f / l_tot, op, a.d);
    // a row that saw nothing but masked keys: see canonical_bias
    if (g == 0)
        a.lse[(int64_t)at.bh * a.sq + i] = m == -kFltMax ? l_tot * kMaskedRowLse
                                                         : row_lse(m, l_tot);
    return true;
}
template <int DB, int kMode, int kWaves, int kHalves>
__global__ __launch_bounds__(kHalves* kWaves * 64, per_simd(DB, kHalves* kWaves)) void
attn_f32_fwd_kernel(const AttnArgs a_in) {
    constexpr int kFwdThreads = kHalves * kWaves * 64, kFwdTile = kHalves * kTile;
    constexpr int kRows = 16 * kWaves;
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    if (kVec ? (kMode & 2) != 0 : a.dropout != 0) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    const Place at(a, a.sq, kRows, true);
    const int limit = (kVec ? (kMode & 1) != 0 : a.has_bias != 0)
                          ? key_bias_span<kFwdThreads, true, false>(a, at.b, at.h, 0, a.sk,
                                                             reinterpret_cast<int*>(lds)).limit
                          : a.sk;
    int j_lo, j_hi;
    key_range(a, at.row0, min(at.row0 + kRows, a.sq), j_lo, j_hi);
    j_hi = max(j_lo + 1, min(j_hi, limit));
    int t_lo = j_lo / kFwdTile, t_hi = (j_hi + kFwdTile - 1) / kFwdTile;
    if (a.n_split > 1) split_tiles(a.n_split, at.split, t_lo, t_hi);
    if (fwd_pass<DB, kMode, kWaves, kHalves, true>(a, at, t_lo, t_hi, lds)) return;
    __syncthreads();
    a = read_again();
    fwd_pass<DB, kMode, kWaves, kHalves, false>(a, Place(a, a.sq, kRows, true), t_lo, t_hi, lds);
}

// dQ: dq_i = scale * sum_j ds_ij k_j,  ds = p (dp - delta),  dp = dO_i . v_j.  Also computes
// delta = rowsum(dO * O) of its rows and stores it for the dK / dV kernel, which runs second.
template <int DB, int kMode, int kWaves, bool kParts>
__device__ __forceinline__ bool dq_pass(const AttnArgs& a, const Place& at, int t_lo, int t_hi,
                                        float* lds) {
    constexpr int kThreads = kWaves * 64, KS = kStepsOf<DB>;
    constexpr bool kVec = kMode != kGeneral;
    constexpr float kLift = lift<kParts>;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    typedef Tile<DB, kVec, kTile, kThreads, kParts> tile_t;
    constexpr int kElems = tile_t::kElems, kPlane = tile_t::kPlane;
    bf16_t* ks = reinterpret_cast<bf16_t*>(lds);
    bf16_t* vs = ks + 2 * kElems;
    const int lane = thread_of<kParts>() & 63, g = lane >> 4, row_g = lane_row(g);
    const int wq0 = at.row0 + 16 * __builtin_amdgcn_readfirstlane(thread_of<kParts>() >> 6);
    const int i = wq0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];
    const float* gp = reinterpret_cast<const float*>(a.dout) + at.b * a.os[0] + at.h * a.os[2];
    const float* op = reinterpret_cast<const float*>(a.o) + at.b * a.os[0] + at.h * a.os[2];

    float top = 0.f;
    tile_t kt, vt;
    operand_t<kParts> qf[KS], gf[KS];
    f32x4_t dq[DB];
    kt.load(kp, a.ks[1], t_lo * kTile, a.sk, a.d);
    vt.load(vp, a.vs[1], t_lo * kTile, a.sk, a.d);
    float delta = 0.f;
    {
        f32x4_t row[2 * KS], out[2 * KS];
        load_row<kParts, kVec, KS>(row, qp, a.qs[1], i, a.sq, a.d, a.scale_log2 / kLift);
        if (kParts) track_row(top, row);
        hold_row<kParts, KS>(qf, row);
        load_row<kParts, kVec, KS>(row, gp, a.os[1], i, a.sq, a.d, 1.0f);
        load_row<kParts, kVec, KS>(out, op, a.os[1], i, a.sq, a.d, 1.0f);
#pragma unroll
        for (int x = 0; x < 2 * KS; ++x) {
#pragma unroll
            for (int e = 0; e < 4; ++e) delta = __builtin_fmaf(out[x][e], row[x][e], delta);
            row[x] *= kLift;
        }
        hold_row<kParts, KS>(gf, row);
        delta = column_sum(delta);
#pragma unroll
        for (int x = 0; x < DB; ++x) dq[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    const float lse_raw = i < a.sq ? a.lse[(int64_t)at.bh * a.sq + i] : 0.f;
    const float lse = lse_reference(lse_raw, kLog2e), inv_n = lse_row_factor(lse_raw);
    const float rest = masked_row_lse(lse_raw) ? 0.f : __builtin_fmaf(lse_raw, -kLog2e, lse);
    if (g == 0 && i < a.sq) a.delta[(int64_t)at.bh * a.sq + i] = delta;
    delta *= kLift;
    kt.template store<kParts, true>(ks, t_lo * kTile, a.sk, a.d, top);
    vt.template store<kParts, true>(vs, t_lo * kTile, a.sk, a.d, top);
    __syncthreads();

    const int wq_last = min(wq0 + 15, a.sq - 1);
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const bf16_t *kb = ks + slot * kElems, *vb = vs + slot * kElems;
        if (kParts && t + 1 < t_hi) {
            kt.load(kp, a.ks[1], (t + 1) * kTile, a.sk, a.d);
            vt.load(vp, a.vs[1], (t + 1) * kTile, a.sk, a.d);
        }
        const int j0 = t * kTile;
        const bool active = wq0 < a.sq && (!a.causal || j0 <= wq_last) &&
                            (a.window <= 0 || wq0 - (j0 + kTile - 1) < a.window);
        if (active) {
            const bool masked = j0 + kTile > a.sk || (a.causal && j0 + kTile - 1 > wq0) ||
                                (a.window > 0 && wq_last - j0 >= a.window);
            uint32_t bits = 0u;
            if (dropout) bits = keep_keys32<kParts>(a, at.bh, i, j0) >> row_g;
            f32x4_t ds[2];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const f32x4_t s = dot_rows<DB, kPlane>(kb, 16 * h2, qf, splat(rest));
                const f32x4_t dp = dot_rows<DB, kPlane>(vb, 16 * h2, gf);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int j = j0 + 16 * h2 + 4 * r + row_g;
                    float x = s[r], y = dp[r];
                    if (has_bias)
                        x += bias_at(a, at.b, at.h, min(i, a.sq - 1), min(j, a.sk - 1));
                    if (dropout) y = (bits >> (16 * h2 + 4 * r)) & 1u ? y * a.rng.inv_keep : 0.f;
                    y = y * (1.0f / kLift) - delta;  // (dO v: kLift^2 times itself)
                    if (has_bias) y *= inv_n;  // (1 without a bias)
                    ds[h2][r] = exp2_of<kParts>(x - lse) * y;
                }
            }
            if (masked) {  // uniform
                const Visible vis = keys_of_query(a, i, j0 + row_g);
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!vis(16 * h2 + 4 * r)) ds[h2][r] = 0.f;
            }
            add_rows<DB, kPlane>(kb, operand<kParts>(ds[0], ds[1]), dq, dq);
        }
        if (t + 1 < t_hi) {
            if (!kParts) kt.load(kp, a.ks[1], (t + 1) * kTile, a.sk, a.d);
            kt.template store<kParts, true>(ks + (slot ^ 1) * kElems, (t + 1) * kTile, a.sk, a.d, top);
            if (!kParts) vt.load(vp, a.vs[1], (t + 1) * kTile, a.sk, a.d);
            vt.template store<kParts, true>(vs + (slot ^ 1) * kElems, (t + 1) * kTile, a.sk, a.d, top);
        }
        __syncthreads();
    }
    if constexpr (kParts) {
        const bool ok = top <= kTop && not_finite(dq) == 0.f;
        if (!everywhere<kWaves>(ok, reinterpret_cast<int*>(lds))) return false;
    }
    if (i >= a.sq) return true;
    if (a.n_split > 1) {
        store_row<kParts, kVec>(dq, 1.0f / (kLift * kLift), a.scale, a.part + (at.part_row0 + i) * a.d, a.d);
        return true;
    }
    float* dqp = reinterpret_cast<float*>(a.dq) + at.b * a.dqs[0] + (int64_t)i * a.dqs[1] +
                 at.h * a.dqs[2];
    store_row<kParts, kVec>(dq, 1.0f / (kLift * kLift), a.scale, dqp, a.d);
    return true;
}
template <int DB, int kMode, int kWaves>
__global__ __launch_bounds__(kWaves * 64, per_simd_bwd(DB, false)) void
attn_f32_dq_kernel(const AttnArgs a_in) {
    constexpr int kThreads = kWaves * 64, kRows = 16 * kWaves;
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    if (kVec ? (kMode & 2) != 0 : a.dropout != 0) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    const Place at(a, a.sq, kRows, true);
    const int limit = (kVec ? (kMode & 1) != 0 : a.has_bias != 0)
                          ? key_bias_span<kThreads, true, false>(a, at.b, at.h, 0, a.sk,
                                                          reinterpret_cast<int*>(lds)).limit
                          : a.sk;
    int j_lo, j_hi;
    key_range(a, at.row0, min(at.row0 + kRows, a.sq), j_lo, j_hi);
    j_hi = max(j_lo + 1, min(j_hi, limit));
    int t_lo = j_lo / kTile, t_hi = (j_hi + kTile - 1) / kTile;
    if (a.n_split > 1) split_tiles(a.n_split, at.split, t_lo, t_hi);
    if (dq_pass<DB, kMode, kWaves, true>(a, at, t_lo, t_hi, lds)) return;
    __syncthreads();
    a = read_again();
    dq_pass<DB, kMode, kWaves, false>(a, Place(a, a.sq, kRows, true), t_lo, t_hi, lds);
}

// dK and dV: a wavefront owns 16 keys, queries stream through LDS.
//   dv_j = sum_i pdrop_ij dO_i          dk_j = scale * sum_i ds_ij q_i
template <int DB, int kMode, int kWaves, bool kParts>
__device__ __forceinline__ bool dkv_pass(const AttnArgs& a, const Place& at, int t_lo, int t_hi,
                                         float* lds) {
    constexpr int kThreads = kWaves * 64, KS = kStepsOf<DB>;
    constexpr bool kVec = kMode != kGeneral;
    constexpr float kLift = lift<kParts>;
    const bool has_bias = kVec ? (kMode & 1) != 0 : a.has_bias != 0;
    const bool dropout = kVec ? (kMode & 2) != 0 : a.dropout != 0;
    typedef Tile<DB, kVec, kTile, kThreads, kParts> tile_t;
    constexpr int kElems = tile_t::kElems, kPlane = tile_t::kPlane;
    bf16_t* qs = reinterpret_cast<bf16_t*>(lds);
    bf16_t* gs = qs + 2 * kElems;
    // [2][4][kTile]: lse reference and its rest, its factor, delta; rows in the order of the accumulators (row
    // 16 h + 4 r + e at 16 h + 4 e + r)
    float* rows = reinterpret_cast<float*>(gs + 2 * kElems);
    const int lane = thread_of<kParts>() & 63, g = lane >> 4, row_g = lane_row(g);
    const int wk0 = at.row0 + 16 * __builtin_amdgcn_readfirstlane(thread_of<kParts>() >> 6);
    const int j = wk0 + (lane & 15);
    const float* qp = reinterpret_cast<const float*>(a.q) + at.b * a.qs[0] + at.h * a.qs[2];
    const float* kp = reinterpret_cast<const float*>(a.k) + at.b * a.ks[0] + at.h * a.ks[2];
    const float* vp = reinterpret_cast<const float*>(a.v) + at.b * a.vs[0] + at.h * a.vs[2];
    const float* gp = reinterpret_cast<const float*>(a.dout) + at.b * a.os[0] + at.h * a.os[2];

    float top = 0.f;
    tile_t qt, gt;
    operand_t<kParts> kf[KS], vf[KS];
    f32x4_t dk[DB], dv[DB];
    float lse_r = 0.f, delta_r = 0.f;  // thread x < kTile: row x of the tile on its way
    auto request = [&](int t) __attribute__((always_inline)) {
        qt.load(qp, a.qs[1], t * kTile, a.sq, a.d);
        gt.load(gp, a.os[1], t * kTile, a.sq, a.d);
        if (thread_of<kParts>() < kTile) {
            const int64_t row = (int64_t)at.bh * a.sq + min(t * kTile + (int)thread_of<kParts>(), a.sq - 1);
            lse_r = a.lse[row];
            delta_r = a.delta[row];
        }
    };
    auto publish = [&](int t, int slot) __attribute__((always_inline)) {
        qt.template store<kParts, true>(qs + slot * kElems, t * kTile, a.sq, a.d, top);
        gt.template store<kParts, true>(gs + slot * kElems, t * kTile, a.sq, a.d, top);
        if (thread_of<kParts>() < kTile) {
            const int x = thread_of<kParts>();
            float* r = rows + slot * 4 * kTile + ((x & 16) | (x & 3) << 2 | (x >> 2 & 3));
            const float lse = lse_reference(lse_r, kLog2e);
            r[0] = lse;
            r[kTile] = masked_row_lse(lse_r) ? 0.f : __builtin_fmaf(lse_r, -kLog2e, lse);
            r[2 * kTile] = delta_r * (kLift * kLift * kLift);  // (as dO v p below)
            r[3 * kTile] = lse_row_factor(lse_r);
        }
    };
    {
        f32x4_t row[2 * KS];
        load_row<kParts, kVec, KS>(row, kp, a.ks[1], j, a.sk, a.d, a.scale_log2 / kLift);
        if (kParts) track_row(top, row);
        hold_row<kParts, KS>(kf, row);
        load_row<kParts, kVec, KS>(row, vp, a.vs[1], j, a.sk, a.d, kLift);
        if (kParts) track_row(top, row);
        hold_row<kParts, KS>(vf, row);
    }
#pragma unroll
    for (int x = 0; x < DB; ++x) dk[x] = dv[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (t_lo < t_hi) {
        request(t_lo);
        publish(t_lo, 0);
    }
    __syncthreads();

    // Above head_dim 64 the keep bits are drawn ahead of the next tile's requests, whose registers they would
    // push out to memory (B2 S900 H8 D96 padded, p 0.1, forward and backward 262 -> 250 us, B2 S512 H8 D128 with
    // a per-query mask and p 0.1 163 -> 147); below, the requests have the time of the drawing (B2 S777 H12 D64
    // padded, p 0.1 269 against 291).
    constexpr bool kDrawFirst = DB > 4;
    auto draw = [&](int first) __attribute__((always_inline)) {
        return keep_queries<kParts>(a, at.bh, first + row_g, wk0);
    };
    const int wk_last = min(wk0 + 15, a.sk - 1);
    const float kept = dropout ? a.rng.inv_keep * kLift : kLift;
    for (int t = t_lo; t < t_hi; ++t) {
        const int slot = (t - t_lo) & 1;
        const bf16_t *qb = qs + slot * kElems, *gb = gs + slot * kElems;
        const float* rb = rows + slot * 4 * kTile;
        const int i0 = t * kTile;
        const bool active = wk0 < a.sk && (!a.causal || i0 + kTile - 1 >= wk0) &&
                            (a.window <= 0 || i0 - wk_last < a.window);
        uint32_t drawn[2] = {0u, 0u};
        if (kDrawFirst && dropout && active) drawn[0] = draw(i0), drawn[1] = draw(i0 + 16);
        if (kParts && t + 1 < t_hi) request(t + 1);
        if (active) {
            const bool masked = i0 + kTile > a.sq || wk0 + 16 > a.sk ||
                                (a.causal && i0 < wk0 + 15) ||
                                (a.window > 0 && i0 + kTile - 1 - wk0 >= a.window);
            f32x4_t pd[2], ds[2];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2) {
                const int r0 = 16 * h2 + 4 * row_g;
                const f32x4_t lse = *reinterpret_cast<const f32x4_t*>(rb + r0);
                const f32x4_t rest = *reinterpret_cast<const f32x4_t*>(rb + kTile + r0);
                const f32x4_t delta = *reinterpret_cast<const f32x4_t*>(rb + 2 * kTile + r0);
                const f32x4_t s = dot_rows<DB, kPlane>(qb, 16 * h2, kf, rest);
                const f32x4_t dp = dot_rows<DB, kPlane>(gb, 16 * h2, vf);
                uint32_t bits = drawn[h2];
                if (!kDrawFirst && dropout) bits = draw(i0 + 16 * h2);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = i0 + 16 * h2 + 4 * r + row_g;
                    float x = s[r];
                    if (has_bias)
                        x += bias_at(a, at.b, at.h, min(i, a.sq - 1), min(j, a.sk - 1));
                    float p = exp2_of<kParts>(x - lse[r]);
                    if (has_bias) p *= rb[3 * kTile + r0 + r];  // (1 without a bias)
                    const float keep = dropout && ((bits >> r) & 1u) == 0 ? 0.f : kept;
                    pd[h2][r] = p * keep;
                    ds[h2][r] = p * (dp[r] * keep - delta[r]);
                }
            }
            if (masked) {  // uniform
                const Visible vis = queries_of_key(a, j, i0 + row_g);
#pragma unroll
                for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (!vis(16 * h2 + 4 * r)) pd[h2][r] = ds[h2][r] = 0.f;
            }
            add_rows<DB, kPlane>(gb, operand<kParts>(pd[0], pd[1]), dv, dv);
            add_rows<DB, kPlane>(qb, operand<kParts>(ds[0], ds[1]), dk, dk);
        }
        if (t + 1 < t_hi) {
            if (!kParts) request(t + 1);
            publish(t + 1, slot ^ 1);
        }
        __syncthreads();
    }
    if constexpr (kParts) {
        const bool ok = top <= kTop && not_finite(dv, not_finite(dk)) == 0.f;
        if (!everywhere<kWaves>(ok, reinterpret_cast<int*>(lds))) return false;
    }
    if (j >= a.sk) return true;
    constexpr float kDownV = 1.0f / (kLift * kLift), kDownK = kDownV * kDownV;
    if (a.n_split > 1) {
        float* part = a.part + (at.part_row0 + j) * a.d;
        store_row<kParts, kVec>(dk, kDownK, a.scale, part, a.d);
        store_row<kParts, kVec>(dv, kDownV, 1.0f,
                                part + (int64_t)a.n_split * a.batch * a.heads * a.sk * a.d, a.d);
        return true;
    }
    float* dkp = reinterpret_cast<float*>(a.dk) + at.b * a.dks[0] + (int64_t)j * a.dks[1] +
                 at.h * a.dks[2];
    float* dvp = reinterpret_cast<float*>(a.dv) + at.b * a.dvs[0] + (int64_t)j * a.dvs[1] +
                 at.h * a.dvs[2];
    store_row<kParts, kVec>(dk, kDownK, a.scale, dkp, a.d);
    store_row<kParts, kVec>(dv, kDownV, 1.0f, dvp, a.d);
    return true;
}
template <int DB, int kMode, int kWaves>
__global__ __launch_bounds__(kWaves * 64, per_simd_bwd(DB, kMode >= 2)) void
attn_f32_dkv_kernel(const AttnArgs a_in) {
    constexpr int kThreads = kWaves * 64, kRows = 16 * kWaves;
    AttnArgs a = a_in;
    constexpr bool kVec = kMode != kGeneral;
    if (kVec ? (kMode & 2) != 0 : a.dropout != 0) resolve_device_state(a.rng);
    extern __shared__ __align__(16) float lds[];
    const Place at(a, a.sk, kRows, false);
    const int limit = (kVec ? (kMode & 1) != 0 : a.has_bias != 0)
                          ? key_bias_span<kThreads, true, false>(a, at.b, at.h, 0, a.sk,
                                                          reinterpret_cast<int*>(lds)).limit
                          : a.sk;
    int i_lo, i_hi;
    query_range(a, at.row0, min(at.row0 + kRows, a.sk), i_lo, i_hi);
    // keys past the last unpadded one get no probability from any row
    if (at.row0 >= limit) i_hi = i_lo;
    int t_lo = i_lo / kTile, t_hi = (i_hi + kTile - 1) / kTile;
    if (a.n_split > 1) split_tiles(a.n_split, at.split, t_lo, t_hi);
    if (dkv_pass<DB, kMode, kWaves, true>(a, at, t_lo, t_hi, lds)) return;
    __syncthreads();
    a = read_again();
    dkv_pass<DB, kMode, kWaves, false>(a, Place(a, a.sk, kRows, false), t_lo, t_hi, lds);
}

enum class Which { kFwd, kDq, kDkv };

// DB = 16-wide blocks of the head dimension
template <int DB, Which kWhich, int kMode, int kWaves, int kHalves = 1>
int launch_build(const AttnArgs& a, hipStream_t st) {
    const int n_rows = kWhich == Which::kDkv ? a.sk : a.sq;
    constexpr int kRows = 16 * kWaves;
    const int64_t blocks =
        (int64_t)((n_rows + kRows - 1) / kRows) * a.batch * a.heads * a.n_split;
    if (blocks <= 0 || blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    const size_t smem = 4 * 3 * kHalves * kTile * kPitchOf<DB> * sizeof(bf16_t) +
                        (kWhich == Which::kDkv ? 8 * kTile * sizeof(float) : 0);
    auto kern = [] {
        if constexpr (kWhich == Which::kFwd) return attn_f32_fwd_kernel<DB, kMode, kWaves, kHalves>;
        else if constexpr (kWhich == Which::kDq) return attn_f32_dq_kernel<DB, kMode, kWaves>;
        else return attn_f32_dkv_kernel<DB, kMode, kWaves>;
    }();
    static std::atomic<uint64_t> lds_ready{0};
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_ready) != SLAPO_OK)
        return SLAPO_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kHalves * kWaves * 64), smem, st, a);
    return check_launch();
}
template <int DB, Which kWhich, int kMode>
int launch(const AttnArgs& a, hipStream_t st) {
    const int n_rows = kWhich == Which::kDkv ? a.sk : a.sq;
    const int64_t units = (int64_t)((n_rows + 63) / 64) * a.batch * a.heads * a.n_split;
    if constexpr (DB > 6) {
        return launch_build<DB, kWhich, kMode, 8>(a, st);
    } else {
        if constexpr (kWhich == Which::kFwd)
            if (units < kHalvesBelow) return launch_build<DB, kWhich, kMode, 4, 2>(a, st);
        if constexpr (DB <= 4)
            if (kWhich == Which::kFwd || units >= kWideBwd)
                return launch_build<DB, kWhich, kMode, 8>(a, st);
        return launch_build<DB, kWhich, kMode, 4>(a, st);
    }
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
