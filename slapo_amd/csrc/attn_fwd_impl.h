// Flash-attention forward for gfx950 (fp16 / bf16 inputs, fp32 accumulation).
//
// One workgroup (4 wavefronts) owns 128 consecutive queries of one (batch, head); wavefront w owns
// 32 of them, lane l = one query (lanes l and l + 32 share a query and split the registers' keys
// resp. head-dim slots).  Keys and values stream through LDS in tiles of 64, double buffered and
// staged through registers (the global loads of tile t+1 are in flight while tile t is
// processed).  Per key tile, as two halves of 32 keys:
//   S^T  = K Q^T                  A = K rows from LDS (row-permuted 128-bit reads), B = Q^T regs
//   P^T  = exp2(S^T * scale - m)  online softmax with a lazily moved reference point m
//   O^T += V^T P^T                B = P^T straight from the accumulator registers (the row
//                                 permutation of the K reads makes them ordered k-slots), A = V^T
//                                 read from the row-major V tile with the transposing LDS read.
// The loop is deliberately NOT software pipelined across tiles inside a wavefront: one tile is in
// flight per wavefront.  Tiles that no query of the workgroup needs masks for come first, as one
// straight block; all others share one body (TileOrder, visible_bits).  That keeps the kernel inside
// 168 registers at head_dim <= 64 (three workgroups per CU; four in 128 without bias and dropout) and
// inside 256 above (two), and on this hardware resident wavefronts hide
// more latency than a deeper pipeline inside one wavefront does: a pipelined variant with twice
// the registers measured 12 % slower at head_dim 64 and 35-80 % slower at 80 / 128.
//
// Launches that leave CUs idle take workgroups of 64 or 32 queries whose wavefronts share the keys (kGroups).
//
// Reference semantics: slapo/op/attention.py:163-181 (attention_bmk), :97-131 (flash_attn_ref).
#pragma once
#include <type_traits>

#include "attn_common.h"

namespace slapo {
namespace fwd {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kBM = kWaves * 32;
constexpr int kBN = 64;
constexpr float kMaxSlack = 8.0f;  // hysteresis of the softmax reference, log2 units

// Workgroups per CU: four in 128 registers up to head_dim 32, three in 168 up to 64, two above (three at 96 spill 2 to 54
// registers: bf16 B2 S3000 H20 D80 padded 147 -> 185 us).
constexpr int fwd_per_cu(int dpad) { return dpad <= 32 ? 4 : dpad <= 64 ? 3 : 2; }
// At 64 without bias and dropout four fit in 128 registers, which pays where the launch fills them: from the
// first workgroup that three a CU would not hold on (fp16 B8 S1024 H16 D64 causal, 1024 workgroups:
// 30.8 -> 29.5 us, bf16 B2 S4096 H16 D64 causal 88.5 -> 83.1; bf16 B1 S8192 H8 D64, 512: 167 -> 169).
constexpr int kFwdFour = 4;

// Small launches: kGroups groups of wavefronts, each with an equal share of the key tiles of the same
// 128 / kGroups queries, merged through LDS at the end.  A launch that leaves CUs idle takes as long as one
// workgroup needs for all its tiles (0.9 us each at head_dim 64, 1.3 at 128, and 4 to start and end), and
// kGroups as many workgroups walk a kGroups-th each.  With four groups a wavefront stages its own tiles
// and meets no barrier.  What it costs is K / V traffic, kGroups times as much from L2.
constexpr int group_rows(int groups) { return kBM / groups; }
// LDS slots of a group's K and of its V tiles: one where a group is a single wavefront, whose LDS accesses
// are in order anyway, or where two would leave one workgroup per CU.
constexpr int group_slots(int groups, int dpad) { return groups == 1 || (groups == 2 && dpad <= 64) ? 2 : 1; }
template <typename T, int DPAD, int kBias, int kGroups>
constexpr size_t group_lds() {
    return (size_t)2 * group_slots(kGroups, DPAD) * kBN * (DPAD + 8) * sizeof(T) +
           (kBias == 2 || kBias == 4 ? 2 * kBN * sizeof(float) : 0);
}
// Workgroups per CU: two where the second hides more than the registers cost that the build spills for it (up
// to 26, at head_dim 65 to 96 with a key mask or bits of any geometry).  One / two per CU, bf16:
//   two groups   D64 B1 S1024 H16 14.1 / 13.1 us; D80 S1024 H8 with a 16-bit key mask 15.3 / 14.7, B4 S512 H16 bits of
//                any geometry 115 / 75.7; with a prepared bias D80 B2 S777 H12 causal 19.8 / 39.2; above 96 S1024 H16
//                24.2 / 23.8, stored bits 25.8 / 27.4, with a prepared bias 36.5 / 49.0
//   four groups  D64 S1024 H16 18.9 / 14.4, with a prepared bias and drawn bits S1024 H8 causal 16.6 / 23.8; D80 S1024
//                H8 with a 16-bit key mask 15.7 / 26.2
constexpr int group_per_cu(int groups, int dpad, int bias) {
    return dpad <= 32 || (groups == 4 ? dpad <= 64 && bias != 3 : dpad <= 64 || (dpad <= 96 && bias != 3))
               ? 2
               : 1;
}

template <typename T, int DPAD, int kBias, int kDrop, int kSteps, int kPerCu, int kGroups>
__global__ __launch_bounds__(kThreads, kPerCu) void attn_fwd_kernel(
    const AttnArgs a_in) {
    // kBias: 0 = no additive bias, 1 = any layout (read from memory per score), 2 = the bias
    // depends on the key only (stride 0 over the queries, e.g. a [B,1,1,Sk] padding mask): the 64
    // values of a key tile travel through LDS beside the K / V tile and the tile body has neither
    // global loads nor branches for them (bf16 B4 S2048 H32 D80 causal, every key valid: 241 us
    // with the per-score reads against 169 us without a bias), 3 = a prepared bias
    // (bias_prepare_kernel): fp32 rows in log2 units, padded and in accumulator order, so that a
    // lane reads its sixteen values of a half with four 16-byte loads and nothing else.
    // 4 = like 2 for a bias of any type (16-bit masks at inference; the selects of the conversion cost
    // the forward 2 %, so that training, whose backward kernels read fp32 anyway, keeps 2).
    constexpr bool kKeyBias = kBias == 2 || kBias == 4;
    AttnArgs a = a_in;
    if constexpr (kDrop == 1 || kDrop == 2) resolve_device_state(a.rng);
    typedef typename Mma<T>::frag frag_t;
    constexpr int kRowWaves = kWaves / kGroups, kRows = group_rows(kGroups);
    constexpr int kSlots = group_slots(kGroups, DPAD);
    typedef TileStage<T, DPAD, kBN, kRowWaves * 64> Stage;
    constexpr int kPitch = Stage::kPitch;
    constexpr int kTileElems = kBN * kPitch;
    // k-steps of S^T = K Q^T: DPAD / 16, or one fewer where the launcher guarantees head_dim <=
    // 16 * kSteps (head_dim 80 in the 96-wide build: the sixth step would multiply zeros)
    constexpr int DK = kSteps;
    constexpr int DV = DPAD / 32;  // 32-row blocks of O^T

    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wavefront-uniform
    const int group = kGroups == 1 ? 0 : wave / kRowWaves;
    const int row_wave = kGroups == 1 ? wave : wave % kRowWaves;
    T* k_lds = reinterpret_cast<T*>(smem_raw + group * group_lds<T, DPAD, kBias, kGroups>());
    T* v_lds = k_lds + kSlots * kTileElems;  // K[kSlots][tile], V[kSlots][tile]
    float* bias_lds = reinterpret_cast<float*>(v_lds + kSlots * kTileElems);  // [2][kBN], kKeyBias

    const int n_bh = a.batch * a.heads;
    const int n_qt = (a.sq + kRows - 1) / kRows;
    int work = work_index(a, (int)blockIdx.x, (int)gridDim.x), split = 0;
    if (kGroups == 1 && a.n_split > 1) {
        split = work / (n_bh * n_qt);
        work -= split * n_bh * n_qt;
    }
    const int bh = work % n_bh;
    const int qt = n_qt - 1 - work / n_bh;  // heaviest (latest) query tiles first
    const int b = bh / a.heads;
    const int h = bh % a.heads;
    const int q0 = qt * kRows;

    const int g = lane >> 5;
    const int i_loc = lane & 31;
    const int wq0 = q0 + row_wave * 32;  // first query of this wavefront
    const int q_row = wq0 + i_loc;

    const T* q_base = reinterpret_cast<const T*>(a.q) + b * a.qs[0] + h * a.qs[2];
    const T* k_base = reinterpret_cast<const T*>(a.k) + b * a.ks[0] + h * a.ks[2];
    const T* v_base = reinterpret_cast<const T*>(a.v) + b * a.vs[0] + h * a.vs[2];

    int j_lo, j_hi;
    key_range(a, q0, min(q0 + kRows, a.sq), j_lo, j_hi);
    int bias_from = j_lo;  // keys before this one have a bias of zero
    if constexpr (kKeyBias) {  // skip the tiles that hold nothing but padded keys
        const KeyBiasSpan span = key_bias_span<kThreads, kBias == 4, true>(a, b, h, j_lo, j_hi,
                                                                     reinterpret_cast<int*>(smem_raw));
        j_hi = span.limit, bias_from = span.zeros;
    }
    int t_lo = j_lo / kBN;
    int t_hi = (j_hi + kBN - 1) / kBN;
    const int n_longest = (t_hi - t_lo + kGroups - 1) / kGroups;  // tiles of the group with most
    if constexpr (kGroups > 1)
        split_tiles(kGroups, group, t_lo, t_hi);
    else if (a.n_split > 1)
        split_tiles(a.n_split, split, t_lo, t_hi);
    const int n_tiles = t_hi - t_lo;
    const TileOrder order = TileOrder::of<kRows, kBN>(a, q0, t_lo, t_hi);
    const int first = order.first() * kBN;  // first key of the first tile

    // Start-up loads, all issued before any is used: the Q^T fragments (column i = this lane's
    // query, k-slots = 8 consecutive head-dim elements) and the first K / V tile.  Addresses are
    // clamped into the tensors; what was clamped is zeroed afterwards.
    Stage ks, vs;
    ks.init(a.ks[1], a.d);
    vs.init(a.vs[1], a.d);
    frag_t qf[DK];
    {
        u32x4_t q_raw[DK];
        const int qr = min(q_row, a.sq - 1);
#pragma unroll
        for (int t = 0; t < DK; ++t)
            q_raw[t] = *reinterpret_cast<const u32x4_t*>(q_base + (int64_t)qr * a.qs[1] +
                                                         min(16 * t + 8 * g, a.d - 8));
        ks.load(k_base, a.ks[1], first, a.sk, a.d);
        vs.load(v_base, a.vs[1], first, a.sk, a.d);
        // Q is multiplied by scale * log2(e) once, here: the scores leave the matrix pipe in log2
        // units and no per-score multiplication is left in the tile body.
#pragma unroll
        for (int t = 0; t < DK; ++t)
            qf[t] = scale_frag<T>(keep_or_zero(q_raw[t], q_row < a.sq && 16 * t + 8 * g < a.d),
                                  a.scale_log2);
    }

    f32x16_t o_acc[DV];
#pragma unroll
    for (int x = 0; x < DV; ++x)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[x][r] = 0.f;
    // Softmax state of this lane's query, in log2 units (Q carries scale * log2(e)): m_run is the
    // reference point of l_run / o_acc (-inf: nothing accumulated yet), moved lazily.
    float m_run = -INFINITY;
    float m_ref = 0.f;  // what the exponentials subtract: m_run, or 0 while m_run is -inf
    float l_run = 0.f;  // this lane's share of the running sum
    // kRefInMma: the matrix pipe subtracts the reference as well.  One more matrix instruction per
    // tile whose A operand is a constant (kRefUnit in k-slot 0, zeros elsewhere) and whose B
    // operand holds -m_ref / kRefUnit in that slot gives the start value of both score
    // accumulators, so that the scores arrive relative to m_ref and a probability is one
    // v_exp_f32.  The reference must then be a number of T: it is rounded to T when it moves (the
    // row's probabilities and their sum share whatever value is subtracted, so the rounding
    // cancels in the output, and the log-sum-exp is formed from the rounded value), kept within
    // T's range (fp16: |m_ref| <= 60000 * 64 log2 units) and away from T's subnormals.
    // Measured: 28 fewer vector instructions per tile (118 -> 90 at head_dim 64) change nothing at
    // head_dim 64 (32.5 us either way at fp16 B8 S1024 H16 causal, 78.7 / 79.2 us with dropout),
    // cost 3 % at head_dim 128 without dropout and 27 % in the window build that reads stored
    // keep bits, and gain 9 % at head_dim 128 where the kernel draws its dropout bits (bf16 B4
    // S2048 H16 causal, p 0.1: 209 -> 190 us): that build has the most live registers, and the
    // subtractions' operands are what it no longer keeps.  Only that build uses it.  (Builds with
    // a bias could not: the masking value -FLT_MAX is no number of T; and the build for the other mask
    // geometries rounds as the one that reads stored bits does, which stands in for it wherever
    // there is a buffer for them.)
    constexpr bool kRefInMma = kBias == 0 && kDrop == 1 && DPAD > 96;
    constexpr float kRefUnit = std::is_same<T, f16_t>::value ? 64.f : 1.f;
    frag_t ones_frag, ref_frag;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones_frag[j] = (T)0.f, ref_frag[j] = (T)0.f;
    if (g == 0) ones_frag[0] = (T)kRefUnit;

    const int wq_last = min(wq0 + 31, a.sq - 1);
    uint64_t drop_row_base = 0;
    if constexpr (kDrop != 0)
        drop_row_base = ((uint64_t)bh * a.sq + (uint64_t)q_row) * (uint64_t)a.sk;
    const float* bias_row = nullptr;
    if constexpr (kBias == 1 || kBias == 3)  // (rows past the end: the last one)
        bias_row = reinterpret_cast<const float*>(a.bias) + b * a.bs[0] + h * a.bs[1] +
                   (int64_t)min(q_row, a.sq - 1) * a.bs[2];
    // kKeyBias: thread (x & 63) carries key j0 + (x & 63) of the requested tile (all four
    // wavefronts alike, so that neither request nor store needs a branch)
    const float* bias_keys = nullptr;
    if constexpr (kBias == 2)
        bias_keys = reinterpret_cast<const float*>(a.bias) + b * a.bs[0] + h * a.bs[1];
    const BiasKeys bias_typed(a, kBias == 4 ? b * a.bs[0] + h * a.bs[1] : 0);
    float bias_stage = 0.f;
    uint32_t bias_raw = 0;
    auto request_bias = [&](int j0) __attribute__((always_inline)) {
        if constexpr (kBias == 2)
            bias_stage = bias_keys[(int64_t)min(j0 + lane, a.sk - 1) * a.bs[3]];
        if constexpr (kBias == 4) bias_raw = bias_typed.raw(min(j0 + lane, a.sk - 1));
    };
    auto store_bias = [&](int slot) __attribute__((always_inline)) {
        if constexpr (kBias == 4) bias_stage = bias_value(a, bias_raw);
        if constexpr (kKeyBias) bias_lds[slot * kBN + row_slot(lane)] = bias_log2(bias_stage);
    };
    const float* bias_tile = bias_lds;  // the slot of the tile in process
    request_bias(first);

    // per-lane LDS offsets (elements) that do not change from tile to tile
    const int k_off = pi_row(i_loc) * kPitch + 8 * g;
    const int v_off = tr_lane_off(lane, kPitch);

    // Wavefront-uniform: does tile t hold any visible key for this wavefront's queries?
    auto tile_active = [&](int t) __attribute__((always_inline)) {
        if (wq0 >= a.sq) return false;
        const int j0 = t * kBN;
        if (a.causal && j0 > wq_last) return false;
        if (a.window > 0 && wq0 - (j0 + kBN - 1) >= a.window) return false;
        return true;
    };
    // kRowsAhead: the prepared bias of a tile is requested when that of the tile before it has been
    // added, so that it waits neither for itself nor, as loads return in order, for the K / V tile
    // requested in between (bf16 B2 S500 H9 with a [B,1,Sq,Sk] mask, its preparation included: D64
    // 23.9 -> 18.3 us, D80 26.1 -> 22.3; B8 S1024 H16 D80 121 -> 112).  Above head_dim 96 its 32
    // registers spill, and elsewhere than at 64 where the kernel draws keep bits as well (p 0.1 D32 37.2
    // -> 41.6 us, D80 42.5 -> 47.6); up to 64 they cost a workgroup per CU (launch).
    constexpr bool kRowsAhead = kBias == 3 && DPAD <= 96 &&
                                (DPAD > 64 || kPerCu < fwd_per_cu(DPAD)) &&
                                (DPAD == 64 || (kDrop != 1 && kDrop != 2));
    f32x4_t bias_ahead[2][4];
    auto request_rows = [&](int j0) __attribute__((always_inline)) {
        if constexpr (kRowsAhead) {
            // (rows are padded to 64 keys; past the last tile the request is wasted)
            const float* p = bias_row + min(j0, (a.sk - 1) & ~63) + 16 * g;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    bias_ahead[kb][r4] = *reinterpret_cast<const f32x4_t*>(p + 32 * kb + 4 * r4);
        }
    };

    // S^T half = K_half Q^T, in log2 units
    auto half_scores = [&](const T* kt, int kb, f32x16_t& s) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
        if constexpr (kRefInMma) s = Mma<T>::mma32(ones_frag, ref_frag, s);
#pragma unroll
        for (int x = 0; x < DK; ++x)
            s = Mma<T>::mma32(lds_frag<T>(kt + kb * 32 * kPitch + k_off + 16 * x), qf[x], s);
    };
    // bias, masks and maximum of one half; mask_tag: 0 = every key visible, 1 = the causal, window
    // and tail bounds, as one bit per key: two instructions per score whatever the bounds are, so
    // that one masked tile body serves every call, 2 = every key visible and with a bias of zero.
    // Returns this lane's maximum.
    auto finish_half = [&](f32x16_t& s, int t, int kb, auto mask_tag)
                           __attribute__((always_inline)) -> float {
        constexpr int kMask = decltype(mask_tag)::value;
        const int j0 = t * kBN + 32 * kb;
        // register r is key j0 + acc_row(r, g) = j0 + kAccGroupStep g + c with c = acc_row(r, 0)
        uint32_t visible = 0u;
        if constexpr (kMask == 1) {
            const int k_max = a.causal ? min(a.sk - 1, q_row) : a.sk - 1;
            const int k_min = a.window > 0 ? q_row - a.window + 1 : 0;
            const int at = j0 + kAccGroupStep * g;
            visible = visible_bits(k_min - at, k_max - at);
        }
        if constexpr (kBias == 1) {
            // Registers 8 h + e and 8 h + 4 + e are keys 2 g and 2 g + 1 of the aligned group of
            // four keys at j0 + 16 h + 4 e: one 16-byte read per group where the layout allows.
#pragma unroll
            for (int he = 0; he < 8; ++he) {
                const int kg = j0 + 16 * (he >> 2) + 4 * (he & 3);
                float b_lo = 0.f, b_hi = 0.f;
                if (a.bias_vec4 && kg + 3 < a.sk) {
                    const f32x4_t t4 = *reinterpret_cast<const f32x4_t*>(bias_row + kg);
                    b_lo = g ? t4.z : t4.x;
                    b_hi = g ? t4.w : t4.y;
                } else {
                    const int k_lo = kg + 2 * g;
                    if (k_lo < a.sk) b_lo = bias_row[(int64_t)k_lo * a.bs[3]];
                    if (k_lo + 1 < a.sk) b_hi = bias_row[(int64_t)(k_lo + 1) * a.bs[3]];
                }
                s[8 * (he >> 2) + (he & 3)] += bias_log2(b_lo);
                s[8 * (he >> 2) + 4 + (he & 3)] += bias_log2(b_hi);
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            if constexpr (kBias == 3) {
                const f32x4_t t4 = kRowsAhead
                                       ? bias_ahead[kb][r4]
                                       : *reinterpret_cast<const f32x4_t*>(bias_row + j0 + 16 * g +
                                                                           4 * r4);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[4 * r4 + e] += t4[e];
            }
            if constexpr (kKeyBias && kMask != 2) {
                const f32x4_t t4 = *reinterpret_cast<const f32x4_t*>(bias_tile + 32 * kb +
                                                                     quad_slot(r4, g));
                s[4 * r4 + 0] += t4.x;
                s[4 * r4 + 1] += t4.y;
                s[4 * r4 + 2] += t4.z;
                s[4 * r4 + 3] += t4.w;
            }
            if constexpr (kMask == 1) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s[4 * r4 + e] = keep_or_hide(s[4 * r4 + e], visible, acc_row(4 * r4 + e, 0));
            }
            mx = fmaxf(mx, fmaxf(fmaxf(s[4 * r4], s[4 * r4 + 1]),
                                 fmaxf(s[4 * r4 + 2], s[4 * r4 + 3])));
        }
        return mx;
    };
    // Moves the reference point if this tile's maximum calls for it (rare after a row's first
    // tile): only when the maximum exceeds it by more than kMaxSlack, so that the rescale of the
    // accumulators stays off the common path.  A row that has met nothing but masked keys
    // sits at -FLT_MAX and moves up to the first real key like any other.
    auto update_reference = [&](float mx, f32x16_t& s0, f32x16_t& s1)
                                __attribute__((always_inline)) {
        if constexpr (!kRefInMma) {
            const bool move = mx > m_run + kMaxSlack && mx != -INFINITY;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(move) != 0, 0)) {
                // exp2(old reference - new reference); an unset reference (-inf) scales by 0
                const float alpha = (m_run == -INFINITY) ? 0.f : fast_exp2(m_run - mx);
                if (move) {
                    m_run = mx;
                    m_ref = mx;
                    l_run *= alpha;
#pragma unroll
                    for (int x = 0; x < DV; ++x)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o_acc[x][r] *= alpha;
                }
            }
        } else {
            // mx is relative to m_ref here (the scores left the matrix pipe that way)
            const bool move = (m_run == -INFINITY) ? mx != -INFINITY : mx > kMaxSlack;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(move) != 0, 0)) {
                // the new reference as a number of T (times kRefUnit), in range and normal
                constexpr float kTop = std::is_same<T, f16_t>::value ? 60000.f : 3.0e38f;
                constexpr float kTiny = std::is_same<T, f16_t>::value ? 6.2e-5f : 1.2e-38f;
                float x = -(m_ref + mx) * (1.0f / kRefUnit);
                x = fminf(fmaxf(x, -kTop), kTop);
                if (fabsf(x) < kTiny) x = 0.f;
                const T xt = (T)x;
                const float m_new = -(float)xt * kRefUnit;
                const float alpha = (m_run == -INFINITY) ? 0.f : fast_exp2(m_run - m_new);
                if (move) {
                    const float shift = m_new - m_ref;  // this tile's scores move with it
#pragma unroll
                    for (int r = 0; r < 16; ++r) s0[r] -= shift, s1[r] -= shift;
                    m_run = m_new;
                    m_ref = m_new;
                    if (g == 0) ref_frag[0] = xt;
                    l_run *= alpha;
#pragma unroll
                    for (int x2 = 0; x2 < DV; ++x2)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o_acc[x2][r] *= alpha;
                }
            }
        }
    };
    // Keep bits of this lane's query for the 32 keys from j0 on (bit j = key j0 + j), drawn here:
    // Philox blocks cover four consecutive keys; the two lanes of a query (l, l ^ 32) draw the
    // blocks of keys 8 g .. 8 g + 7 of each 16-key group and exchange them.
    // Where the 32 rows of the wavefront lie within one call of the generator (all but a few: a call
    // covers 4 T elements), what the call's blocks share sits in scalar registers (PhiloxCall).
    bool one_call = false;
    PhiloxCall call = {};
    uint32_t row_thread = 0;
    if constexpr (kDrop == 1) {
        const uint64_t first = ((uint64_t)bh * a.sq + (uint64_t)min(wq0, a.sq - 1)) * (uint64_t)a.sk >> 2;
        const uint64_t last = (((uint64_t)bh * a.sq + (uint64_t)wq_last + 1) * (uint64_t)a.sk - 1) >> 2;
        one_call = philox_call_fits(a.rng) && first >> a.rng.t_shift == last >> a.rng.t_shift;
        call = philox_call(a.rng.base_counter + (first >> a.rng.t_shift), a.rng.key0, a.rng.key1);
        row_thread = (uint32_t)(drop_row_base >> 2) & (uint32_t)(a.rng.total_threads - 1);
    }
    auto draw_half = [&](int j0) __attribute__((always_inline)) -> uint32_t {
        uint32_t mine = 0;
        if constexpr (kDrop == 1) {
            if (__builtin_expect(one_call, 1)) {
#pragma unroll
                for (int h2 = 1; h2 >= 0; --h2) {
                    const uint32_t thread = row_thread + (uint32_t)(j0 + 16 * h2 + 8 * g) / 4;
                    uint32_t bits = push_keep4(0u, philox_block(call, thread + 1), a.rng.keep_max);
                    bits = push_keep4(bits, philox_block(call, thread), a.rng.keep_max);
                    mine = mine << 16 | bits;
                }
                return or_xor32(mine << (8 * g));
            }
        }
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
            const int pos = 16 * (blk >> 1) + 8 * g + 4 * (blk & 1);
            const int key0 = j0 + pos;
            uint32_t bits = 0;
            if (q_row < a.sq && key0 < a.sk) {
                const uint64_t e0 = drop_row_base + (uint64_t)key0;
                if constexpr (kDrop == 1)
                    bits = dropout_keep4_pow2(a.rng, e0 >> 2);
                else
                    bits = dropout_keep_any(a.rng, e0, min(4, a.sk - key0));
            }
            mine |= bits << pos;
        }
        return or_xor32(mine);
    };
    // probabilities of one half: exp2, dropout, pack to T, row sum
    // (drop_bits: the keep bits of this lane's query for the 32 keys of the half; kDrop == 3
    // passes in the word that keep_mask_kernel stored, the other modes return the drawn one)
    auto half_prob = [&](f32x16_t& s, int t, int kb, uint32_t (&pw)[8], uint32_t& drop_bits)
                         __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = fast_exp2(kRefInMma ? s[r] : s[r] - m_ref);
        if constexpr (kDrop != 0) {
            float psum = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) psum += s[r];
            l_run += psum;
            uint32_t mine = drop_bits;
            if constexpr (kDrop != 3) mine = draw_half(t * kBN + 32 * kb);
            const uint32_t mine_g = mine >> (kAccGroupStep * g);
            // dropped probabilities become +0 (two instructions each); the factor 1 / (1 - p) of
            // the kept ones goes onto the output rows when they are written
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = keep_or_zero(s[r], mine_g, acc_row(r, 0));
            drop_bits = mine;
#pragma unroll
            for (int r2 = 0; r2 < 8; ++r2) pw[r2] = pack2<T>(s[2 * r2], s[2 * r2 + 1]);
        } else {
            // Without dropout the row sum is taken over the rounded probabilities, two per
            // instruction (v_dot2c_f32_{f16,bf16} against a pair of ones): the normaliser then
            // belongs to exactly the numbers that multiply V.
#pragma unroll
            for (int r2 = 0; r2 < 8; ++r2) {
                pw[r2] = pack2<T>(s[2 * r2], s[2 * r2 + 1]);
                l_run = sum2<T>(pw[r2], l_run);
            }
        }
    };
    // O^T += V_half^T P_half^T
    auto half_accumulate = [&](const T* vt, int kb, const uint32_t (&pw)[8])
                               __attribute__((always_inline)) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            u32x4_t pq = {pw[4 * s2], pw[4 * s2 + 1], pw[4 * s2 + 2], pw[4 * s2 + 3]};
            const frag_t pf = __builtin_bit_cast(frag_t, pq);
#pragma unroll
            for (int x = 0; x < DV; ++x)
                o_acc[x] = Mma<T>::mma32(
                    lds_frag_tr<T>(vt + (32 * kb + 16 * s2) * kPitch + v_off + 32 * x, kPitch), pf,
                    o_acc[x]);
        }
    };
    // kDrop == 3: the keep bits of this lane's query for the two halves of a tile, drawn by
    // keep_mask_kernel.  Requested a tile ahead and before the tile's K / V: loads return in order, so
    // that a word requested after them would make the probabilities wait for the whole next tile.
    uint32_t tile_bits[2] = {0u, 0u}, next_bits[2] = {0u, 0u};
    auto request_bits = [&](int t) __attribute__((always_inline)) {
        if constexpr (kDrop == 3) {
            const int64_t base = (int64_t)bh * a.mask_words;
            const int row = min(q_row, a.sq - 1);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                next_bits[kb] =
                    a.keep_mask[(base + min(2 * t + kb, a.mask_words - 1)) * a.mask_pitch + row];
        }
    };
    auto tile_body = [&](const T* kt, const T* vt, int t, int next, auto mask_tag)
                         __attribute__((always_inline)) {
        f32x16_t s0, s1;
        uint32_t pw0[8], pw1[8];
        uint32_t bits0 = 0, bits1 = 0;
        if constexpr (kDrop == 3) bits0 = tile_bits[0], bits1 = tile_bits[1];
        half_scores(kt, 0, s0);
        half_scores(kt, 1, s1);
        const float mx =
            max_xor32(fmaxf(finish_half(s0, t, 0, mask_tag), finish_half(s1, t, 1, mask_tag)));
        request_rows(next);
        update_reference(mx, s0, s1);
        half_prob(s0, t, 0, pw0, bits0);
        half_accumulate(vt, 0, pw0);
        half_prob(s1, t, 1, pw1, bits1);
        half_accumulate(vt, 1, pw1);
        // With dropout and a keep_mask buffer: one word per query and half for the backward.
        // The (wavefront-uniform) branch sits at the end of the tile, where the basic block ends
        // anyway; inside the body it would keep the scheduler from mixing the Philox arithmetic
        // with the matrix instructions (10 % of the forward).
        if constexpr (kDrop == 1 || kDrop == 2) {
            if (a.keep_mask != nullptr) {
                const uint32_t w0 = bits0, w1 = bits1;  // already combined over the lane pair
                uint32_t* row = a.keep_mask +
                                ((int64_t)bh * a.mask_words + 2 * t) * a.mask_pitch + q_row;
                if (g == 0 && q_row < a.sq) {
                    if (t * kBN < a.sk) row[0] = w0;
                    if (t * kBN + 32 < a.sk) row[a.mask_pitch] = w1;
                }
            }
        }
    };

    // ---- prologue: tile 0 into LDS ----
    ks.fix(first, a.sk, a.d, 16 * DK);
    vs.fix(first, a.sk, a.d, 16 * DK);
    // The wavefronts of a group see each other's stores to LDS (all of the workgroup where there are two
    // groups: they walk the same number of barriers).
    auto group_sync = [&]() __attribute__((always_inline)) {
        if constexpr (kRowWaves > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    };
    ks.store(k_lds);
    vs.store(v_lds);
    store_bias(0);
    group_sync();

    // Iteration r: request the next tile, process tile r of the order, write the next tile into the
    // other slot.  kMask != 1: tiles that every wavefront of the workgroup sees in full.
    int t = order.first();
    request_bits(t);
    request_rows(t * kBN);
    auto iteration = [&](int r, auto mask_tag) __attribute__((always_inline)) {
        constexpr bool kFast = decltype(mask_tag)::value != 1;
        const int t_next = kFast ? order.after_fast(t) : order.after(t), next = t_next * kBN;
        const bool have_next = r + 1 < n_tiles;
        tile_bits[0] = next_bits[0], tile_bits[1] = next_bits[1];
        request_bits(t_next);
        // the next tile is requested unconditionally (rows are clamped into the tensor; after the
        // last tile the request is wasted) so that it stays straight-line code.  Requesting it
        // later in the body saves no registers and measures slower.  (Addresses: a scalar tile
        // base plus a per-lane 32-bit offset that is selected, not multiplied out: 2 % faster than
        // the multiplied-out form now that the tile body has no other address arithmetic.)
        ks.load(k_base, a.ks[1], next, a.sk, a.d);
        vs.load(v_base, a.vs[1], next, a.sk, a.d);
        request_bias(next);
        const T* kt = k_lds + (r & (kSlots - 1)) * kTileElems;
        const T* vt = v_lds + (r & (kSlots - 1)) * kTileElems;
        bias_tile = bias_lds + (r & 1) * kBN;
        if constexpr (kFast) {
            tile_body(kt, vt, t, next, mask_tag);
        } else {
            if (tile_active(t))
                tile_body(kt, vt, t, next, mask_tag);
            else
                request_rows(next);
        }
        if constexpr (kSlots == 1) group_sync();
        if (have_next) {
            ks.fix(next, a.sk, a.d, 16 * DK);
            vs.fix(next, a.sk, a.d, 16 * DK);
            ks.store(k_lds + ((r + 1) & (kSlots - 1)) * kTileElems);
            vs.store(v_lds + ((r + 1) & (kSlots - 1)) * kTileElems);
            store_bias((r + 1) & 1);
        }
        group_sync();
        t = t_next;
    };
    int r = 0;
    if constexpr (kKeyBias) {
        // a padding mask is zero up to the padding: no bias to add there, 32 additions and 8 LDS reads
        // of a tile (with key_bias_span, bf16 B2 S7744 H7 D64 at inference 371 -> 339 us, B8 S1024 H16
        // D64 causal 38.6 -> 35.0; as a loop of its own it costs no registers)
        const int zeros = min(order.end, bias_from / kBN) - order.begin;
        for (; r < zeros; ++r) iteration(r, std::integral_constant<int, 2>{});
    }
    for (; r < order.end - order.begin; ++r) iteration(r, std::integral_constant<int, 0>{});
    for (; r < n_tiles; ++r) iteration(r, std::integral_constant<int, 1>{});

    // ---- epilogue ----
    if constexpr (kGroups > 1) {
        if constexpr (kRowWaves > 1)
            for (; r < n_longest; ++r) {  // (the other group's barriers)
                if constexpr (kSlots == 1) group_sync();
                group_sync();
            }
        // The first group adds up: the others leave m, l and O^T in LDS as they sit in registers, a word
        // of 64 lanes after the other.
        constexpr int kWords = 16 * DV + 2;
        float* mine = reinterpret_cast<float*>(smem_raw) + row_wave * (kGroups - 1) * 64 * kWords + lane;
        __syncthreads();
        if (group > 0) {
            float* p = mine + (group - 1) * 64 * kWords;
            p[0] = m_run, p[64] = l_run;
#pragma unroll
            for (int x = 0; x < DV; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e) p[64 * (2 + 16 * x + e)] = o_acc[x][e];
        }
        __syncthreads();
        if (group > 0) return;
        float m = m_run;
#pragma unroll
        for (int k = 0; k < kGroups - 1; ++k) m = fmaxf(m, mine[k * 64 * kWords]);
        // (an unset reference weighs nothing)
        auto weight = [&](float mk) __attribute__((always_inline)) {
            return mk == -INFINITY ? 0.f : fast_exp2(mk - m);
        };
        const float w0 = weight(m_run);
        l_run *= w0;
#pragma unroll
        for (int x = 0; x < DV; ++x)
#pragma unroll
            for (int e = 0; e < 16; ++e) o_acc[x][e] *= w0;
#pragma unroll
        for (int k = 0; k < kGroups - 1; ++k) {
            const float* p = mine + k * 64 * kWords;
            const float w = weight(p[0]);
            l_run = __builtin_fmaf(p[64], w, l_run);
#pragma unroll
            for (int x = 0; x < DV; ++x)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    o_acc[x][e] = __builtin_fmaf(p[64 * (2 + 16 * x + e)], w, o_acc[x][e]);
        }
        m_run = m;
    }
    const float l_tot = sum_xor32(l_run);
    if (kGroups == 1 && a.n_split > 1) {
        const int64_t rows = (int64_t)n_bh * a.sq;
        const int64_t row0 = (int64_t)bh * a.sq + wq0;
        if (wq0 < a.sq)
            store_partial<DPAD>(o_acc, 1.0f, a.part + (split * rows + row0) * a.d, a.sq - wq0, a.d);
        if (q_row < a.sq && g == 0) {
            float* ml = a.part + a.n_split * rows * a.d + 2 * (split * rows + row0 + i_loc);
            ml[0] = m_run, ml[1] = l_tot;
        }
        return;
    }
    const float inv_l = kDrop != 0 ? a.rng.inv_keep / l_tot : 1.0f / l_tot;
    // every wavefront is past the last barrier of the loop: the K buffers are free, and each
    // wavefront routes its 32 output rows through its own quarter of them (with groups: through what the
    // others left for it, which it has read)
    if (wq0 < a.sq) {
        T* o_row0 = reinterpret_cast<T*>(a.o) + b * a.os[0] + (int64_t)wq0 * a.os[1] + h * a.os[2];
        T* rows_lds = reinterpret_cast<T*>(smem_raw);
        if constexpr (kGroups == 1)
            rows_lds += wave * 32 * kPitch;
        else
            rows_lds += row_wave * (kGroups - 1) * 64 * (16 * DV + 2) * 2;
        store_block_via_lds<T, DPAD, kPitch>(o_acc, inv_l, rows_lds, o_row0, a.os[1], a.sq - wq0, a.d);
    }
    if (q_row < a.sq) {
        // A row that met nothing but masked keys (bias_log2) sits at -FLT_MAX with l_tot = their
        // number: the row sum goes out in place of the log-sum-exp, scaled by 2^100.
        if (g == 0)
            a.lse[(int64_t)bh * a.sq + q_row] = m_run == -kFltMax
                                                    ? l_tot * kMaskedRowLse
                                                    : (m_run + __builtin_log2f(l_tot)) * kLn2;
    }
}

template <typename T, int DPAD, int kBias, int kDrop, int kSteps, int kPerCu = fwd_per_cu(DPAD),
          int kGroups = 1>
int launch(const AttnArgs& a, hipStream_t st) {
    const size_t smem = kGroups * group_lds<T, DPAD, kBias, kGroups>();
    const int n_qt = (a.sq + group_rows(kGroups) - 1) / group_rows(kGroups);
    const int64_t blocks = (int64_t)n_qt * a.batch * a.heads * a.n_split;
    if (blocks <= 0 || blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    if constexpr (kGroups == 1 && kBias != 1) {
        const int64_t keys = a.window > 0 ? min(a.sk, a.window + kBM) : a.sk;
        constexpr BiasKind kKind = kBias == 0 ? kNoBias : kBias == 3 ? kPreparedBias : kKeyBias;
        const int groups = a.n_split > 1 ? 1
                                         : attn_fwd_groups(blocks, a.n_cus, (keys + kBN - 1) / kBN, a.d,
                                                           a.causal && a.window <= 0, kKind, kDrop);
        if (groups == 4)
            return launch<T, DPAD, kBias, kDrop, kSteps, group_per_cu(4, DPAD, kBias), 4>(a, st);
        if (groups == 2)
            return launch<T, DPAD, kBias, kDrop, kSteps, group_per_cu(2, DPAD, kBias), 2>(a, st);
    }
    // kRowsAhead against one workgroup more per CU (bf16 B8 S1024 H16, 1024 workgroups): without the
    // causal mask D64 100.8 -> 96.7 us, D32 98.5 -> 95.9; with it, whose workgroups differ in length,
    // 65.8 -> 66.3 and 60.0 -> 64.5, so there only in launches that need not the one more
    if constexpr (kGroups == 1 && DPAD <= 64 && kBias == 3 && kPerCu == fwd_per_cu(DPAD) &&
                  (DPAD == 64 || (kDrop != 1 && kDrop != 2))) {
        if (!a.causal || blocks <= (int64_t)(kPerCu - 1) * a.n_cus)
            return launch<T, DPAD, kBias, kDrop, kSteps, kPerCu - 1>(a, st);
    }
    if constexpr (kGroups == 1 && DPAD <= 64 && kBias == 0 && kDrop == 0 && kPerCu < kFwdFour) {
        if (blocks > (int64_t)kPerCu * a.n_cus)
            return launch<T, DPAD, kBias, kDrop, kSteps, kFwdFour>(a, st);
    }
    auto kern = attn_fwd_kernel<T, DPAD, kBias, kDrop, kSteps, kPerCu, kGroups>;
    static std::atomic<uint64_t> lds_ready{0};  // per instantiation, one bit per device
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_ready) != SLAPO_OK)
        return SLAPO_ERR_LAUNCH;
    AttnArgs ordered = a;
    // (head groups: not where the kernel draws or applies dropout bits -- its workgroups run twice as
    // long there and a group's late heavy ones become the tail: 314 -> 350 us at bf16 B4 S2048 H32
    // D80 causal, p 0.1, 588 -> 667 us at fp16 B2 S4096 H32 D96)
    if (a.n_split == 1)
        set_dispatch_order(&ordered, blocks, kPerCu, kDrop == 0);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), smem, st, ordered);
    return check_launch();
}

template <typename T, int DPAD, int kBias, int kSteps>
int dispatch_drop(const AttnArgs& a, hipStream_t st) {
    if (a.dropout == 1) return launch<T, DPAD, kBias, 1, kSteps>(a, st);
    if (a.dropout == 2) return launch<T, DPAD, kBias, 2, kSteps>(a, st);
    if (a.dropout == 3) return launch<T, DPAD, kBias, 3, kSteps>(a, st);
    return launch<T, DPAD, kBias, 0, kSteps>(a, st);
}
template <typename T, int DPAD, int kSteps = DPAD / 16>
int dispatch_flags(const AttnArgs& a, hipStream_t st) {
    if (!a.has_bias) return dispatch_drop<T, DPAD, 0, kSteps>(a, st);
    if (a.bias_type == SLAPO_BIAS_PREPARED) return dispatch_drop<T, DPAD, 3, kSteps>(a, st);
    // one value per key of a 16-bit type, no dropout (checked by the caller)
    if (a.bias_type != SLAPO_F32) return launch<T, DPAD, 4, 0, kSteps>(a, st);
    return a.bs[2] == 0 ? dispatch_drop<T, DPAD, 2, kSteps>(a, st)  // it depends on the key only
                        : dispatch_drop<T, DPAD, 1, kSteps>(a, st);
}

template <typename T>
int dispatch(const AttnArgs& a, hipStream_t st) {
    // (head_dim 32 in the 64-wide kernels multiplies zeros half the time and holds them in registers and
    // LDS; forward and backward fp16 B8 S1024 H16 D32 causal 110 -> 82 us, bf16 B2 S4096 310 -> 214)
    if (a.d <= 32) return dispatch_flags<T, 32>(a, st);
    if (a.d <= 64) return dispatch_flags<T, 64>(a, st);
    if (a.d <= 80) return dispatch_flags<T, 96, 5>(a, st);  // five k-steps cover head_dim 80
    if (a.d <= 96) return dispatch_flags<T, 96>(a, st);
    if (a.d <= 128) return dispatch_flags<T, 128>(a, st);
    return SLAPO_ERR_SHAPE;
}

}  // namespace fwd
}  // namespace slapo
