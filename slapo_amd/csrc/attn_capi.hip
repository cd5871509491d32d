// C-ABI entry points of the attention path: argument validation, kernel selection (MFMA kernels
// for fp16 / bf16 and for fp32) and the kernel that draws dropout masks ahead of the forward.
#include <algorithm>
#include <mutex>

#include "attn_common.h"

namespace slapo {
int attn_fwd_mfma_f16(const AttnArgs& a, hipStream_t st);
int attn_fwd_mfma_bf16(const AttnArgs& a, hipStream_t st);
int attn_bwd_mfma_f16(const AttnArgs& a, hipStream_t st);
int attn_bwd_mfma_bf16(const AttnArgs& a, hipStream_t st);
int attn_bwd_dq_mfma_f16(const AttnArgs& a, hipStream_t st);
int attn_bwd_dq_mfma_bf16(const AttnArgs& a, hipStream_t st);
int attn_bwd_both_mfma_f16(const AttnArgs& a, hipStream_t st);
int attn_bwd_both_mfma_bf16(const AttnArgs& a, hipStream_t st);
int attn_fwd_f32(const AttnArgs& a, hipStream_t st);
int attn_bwd_dq_f32(const AttnArgs& a, hipStream_t st);
int attn_bwd_f32(const AttnArgs& a, hipStream_t st);
int attn_splits(int64_t blocks, int64_t cus, int64_t tiles, bool f32, bool causal);
int attn_merge_fwd(const AttnArgs& a, int dtype, hipStream_t st);
int attn_merge_bwd(const AttnArgs& a, int dtype, const float* dq_part, int n_dq,
                   const float* dkv_part, int n_dkv, hipStream_t st);
int attn_decode_shares(int64_t n_bh, int n_keys);
int attn_decode(const AttnArgs& a, int dtype, int n_shares, float* part, hipStream_t st);
}  // namespace slapo

using namespace slapo;

namespace {

// Dropout keep bits of a 16-bit attention call, drawn once for the forward and both backward
// kernels: thread (row i, word w) draws the eight Philox blocks of keys 32 w .. 32 w + 31 of
// query i and stores them as one word, keep_mask[(bh * mask_words + w) * mask_pitch + i], bit j =
// keep(i, 32 w + j).  The matrix kernels then only test bits; drawing inside the forward kernel
// costs about fifty vector-ALU cycles per score (47 instructions per block of four) beside
// thirty-two (head_dim 128) or sixteen (64) of matrix work.  Only words that hold a key the row itself can see are drawn: the kernels read
// whole words of every 64-key tile that some query of a 32-query group sees, but a bit that
// belongs to a pair outside the row's own mask meets a probability of zero, so what such words
// hold does not matter and they are left as they are.  With a local window the word columns count
// from the first word of the row's window (under a causal mask window / 32 + 2 of them, not seqlen_k /
// 32: every thread then has a word to draw); without one they are the words themselves.
// kExact: any launch geometry of the dropout plan and any seqlen_k (dropout_keep_run).  Drawn per
// word this costs 9 Philox blocks per 32 scores where the forward kernel, whose lanes hold single
// groups of four, drew one block per score: bf16 B3 S777 H12 D64 without a causal mask, p 0.1,
// forward and backward 199 us before, 89 us with this kernel ahead of the forward.  The words of
// padded keys are left as they are too where the other kernels skip their tiles (a third of them in
// that call's mask).  Units of 64 rows and a word, dealt to the wavefronts one after the other: blocks
// of 256 rows left a quarter of the launch to nine rows at S777.  That call: 22.1 -> 17.3 us (14.1 with PhiloxCall).
template <bool kExact>
__global__ __launch_bounds__(256) void keep_mask_kernel(const AttnArgs a_in, int words) {
    AttnArgs a = a_in;
    resolve_device_state(a.rng);
    // a wavefront owns 64 rows and one of the `words` word columns
    const int lane = threadIdx.x & 63;
    const int unit = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = unit / words * 64 + lane;
    const int bh = blockIdx.y;
    int w = unit % words;
    if (a.has_bias && a.bs[2] == 0 && a.window <= 0) {  // (of type fp32: see set_bias)
        // from the first tile on that holds nothing but padded keys: not read (key_bias_span)
        const float* row = reinterpret_cast<const float*>(a.bias) + bh / a.heads * a.bs[0] +
                           bh % a.heads * a.bs[1];
        bool padded = row[0] > kMaskedBias;  // uniform
        for (int j0 = 64 * (w >> 1); padded && j0 < a.sk; j0 += 64) {
            const int j = min(j0 + lane, a.sk - 1);
            padded = __builtin_amdgcn_ballot_w64(row[(int64_t)j * a.bs[3]] > kMaskedBias) == 0;
        }
        if (padded) return;
    }
    if (i >= a.sq) return;
    if (a.window > 0) w += max(i - a.window + 1, 0) >> 5;
    if (w >= a.mask_words) return;
    if (a.window > 0) {
        if (a.causal && 32 * w > i) return;
        if (i - (32 * w + 31) >= a.window) return;
    } else if (a.causal && 64 * (w >> 1) > (i | 31)) {
        return;  // (without a window: every word of a 64-key tile that the row's group visits)
    }
    const uint64_t row_base = ((uint64_t)bh * a.sq + (uint64_t)i) * (uint64_t)a.sk;
    const uint64_t elem = row_base + 32 * (uint64_t)w;
    const uint32_t word = dropout_keep_run<32, !kExact>(a.rng, elem);
    a.keep_mask[((int64_t)bh * a.mask_words + w) * a.mask_pitch + i] = word;
}

// (grid limit of keep_mask_kernel: one grid row per head; 2^31 / 4 units of 64 rows and a word)
bool keep_mask_kernel_fits(const AttnArgs& a) {
    return (int64_t)a.batch * a.heads <= 65535 &&
           (int64_t)((a.sq + 63) / 64) * a.mask_words < 0x7FFFFFF0;
}
int draw_keep_mask(const AttnArgs& a, hipStream_t st) {
    const int64_t bh = (int64_t)a.batch * a.heads;
    if (!keep_mask_kernel_fits(a)) return SLAPO_ERR_SHAPE;
    // with a window: the words of a row's own window (it spans window / 32 + 1 words at most), and where
    // nothing hides the keys behind the query, those as well
    const int words =
        a.window > 0 && a.causal ? min(a.mask_words, a.window / 32 + 2) : a.mask_words;
    const int units = (a.sq + 63) / 64 * words;
    const dim3 grid((unsigned)((units + 3) / 4), (unsigned)bh);
    if (a.dropout == 1)
        hipLaunchKernelGGL(keep_mask_kernel<false>, grid, dim3(256), 0, st, a, words);
    else
        hipLaunchKernelGGL(keep_mask_kernel<true>, grid, dim3(256), 0, st, a, words);
    return check_launch();
}

// Compute units of the current device (0 if the runtime will not say), asked once per device.
int cus_of_current_device() {
    static std::atomic<int> known[64];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int n = known[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        known[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

bool strides_ok(const int64_t s[3], int mult) {
    return s[0] % mult == 0 && s[1] % mult == 0 && s[2] % mult == 0;
}

int fill_args(const slapo_attn_params* p, AttnArgs* a, bool backward) {
    if (!p) return SLAPO_ERR_ARG;
    if (p->batch <= 0 || p->heads <= 0 || p->seqlen_q <= 0 || p->seqlen_k <= 0 ||
        p->head_dim <= 0)
        return SLAPO_ERR_SHAPE;
    if (p->head_dim > 128) return SLAPO_ERR_SHAPE;
    if ((int64_t)p->batch * p->heads > 0x7FFFFFFF / 2) return SLAPO_ERR_SHAPE;
    if (!(p->p_drop >= 0.f && p->p_drop <= 1.f)) return SLAPO_ERR_ARG;
    if (p->window < 0) return SLAPO_ERR_ARG;
    // the scale is folded into Q / K fragments: a NaN or infinite one would poison every score
    if (!(p->scale > -kFltMax && p->scale < kFltMax)) return SLAPO_ERR_ARG;
    const bool half = p->dtype == SLAPO_F16 || p->dtype == SLAPO_BF16;
    if (!half && p->dtype != SLAPO_F32) return SLAPO_ERR_DTYPE;
    if (half) {
        if (p->head_dim % 8 != 0) return SLAPO_ERR_SHAPE;
        if (!strides_ok(p->q_strides, 8) || !strides_ok(p->k_strides, 8) ||
            !strides_ok(p->v_strides, 8) || !strides_ok(p->o_strides, 8))
            return SLAPO_ERR_ALIGN;
        // the tile loads address rows with 32-bit byte offsets from a per-tile base
        for (const int64_t* st : {p->q_strides, p->k_strides, p->v_strides, p->o_strides})
            if (st[1] < 0 || st[1] >= (int64_t(1) << 24)) return SLAPO_ERR_SHAPE;
    }
    for (int i = 0; i < 3; ++i) {
        a->qs[i] = p->q_strides[i];
        a->ks[i] = p->k_strides[i];
        a->vs[i] = p->v_strides[i];
        a->os[i] = p->o_strides[i];
    }
    for (int i = 0; i < 4; ++i) a->bs[i] = p->bias_strides[i];
    a->batch = p->batch;
    a->heads = p->heads;
    a->sq = p->seqlen_q;
    a->sk = p->seqlen_k;
    a->d = p->head_dim;
    a->causal = p->causal ? 1 : 0;
    a->window = p->window;
    a->scale = p->scale;
    a->scale_log2 = p->scale * kLog2e;
    a->dropout = p->p_drop > 0.f ? 1 : 0;
    if (a->dropout) {
        const int64_t numel = (int64_t)p->batch * p->heads * p->seqlen_q * p->seqlen_k;
        if (!plan_ok(&p->plan, numel)) return SLAPO_ERR_ARG;
        a->rng = make_dropout_state(p->plan, (double)p->p_drop, p->seed, p->offset);
        if (!(a->rng.g_shift >= 0 && a->rng.t_shift >= 0 && p->seqlen_k % 4 == 0)) a->dropout = 2;
    } else {
        a->rng = DropoutState{};
    }
    a->snake_len = 0, a->snake_rows = 0;
    a->n_cus = half ? cus_of_current_device() : 0;
    a->n_split = 1;
    a->part = nullptr;
    a->keep_mask = nullptr;
    a->mask_words = (p->seqlen_k + 31) / 32;
    a->mask_pitch = (p->seqlen_q + 3) & ~3;
    if (a->dropout && half && p->keep_mask) {
        if (!aligned16(p->keep_mask)) return SLAPO_ERR_ALIGN;
        a->keep_mask = reinterpret_cast<uint32_t*>(p->keep_mask);
        if (backward) a->dropout = 3;
    }
    return SLAPO_OK;
}

// The additive bias of a call: SLAPO_ERR_DTYPE for a type that its layout is not read in.
int set_bias(AttnArgs* a, const void* bias, int type, bool f32, bool backward) {
    a->bias = bias;
    a->has_bias = bias ? 1 : 0;
    a->bias_vec4 = 0;
    a->bias_type = type;
    if (!bias) return SLAPO_OK;
    if (a->sq == 1 && type != SLAPO_BIAS_PREPARED) a->bs[2] = 0;
    if (type == SLAPO_BIAS_PREPARED) {
        if (f32) return SLAPO_ERR_DTYPE;
        return aligned16(bias) ? SLAPO_OK : SLAPO_ERR_ALIGN;
    }
    if (type != SLAPO_F32 && type != SLAPO_F16 && type != SLAPO_BF16) return SLAPO_ERR_DTYPE;
    if (type != SLAPO_F32 && !f32) {
        // 16-bit biases of the 16-bit kernels: one value per key in a forward without dropout, or
        // prepared
        if (backward || a->dropout || a->bs[2] != 0) return SLAPO_ERR_DTYPE;
        // (addressed with 32-bit offsets: BiasKeys)
        if (a->bs[3] < 0 || a->bs[3] * a->sk >= int64_t(1) << 30) return SLAPO_ERR_SHAPE;
    }
    if (a->bs[3] == 1 && aligned16(bias) && a->bs[0] % 4 == 0 && a->bs[1] % 4 == 0 &&
        a->bs[2] % 4 == 0)
        a->bias_vec4 = 1;
    return SLAPO_OK;
}

// Additive bias with values of its own per query -> fp32 rows in log2 units, masking values
// canonical, rows and row length padded to 64 with zeros, the keys of a 32-key block in
// accumulator order (prepared_slot).  One thread per four slots; bound by reading the mask and
// writing the rows once (bf16 [B,1,Sq,Sk]: 6 bytes per value), which stands in for the conversion
// to fp32 that such a mask would need anyway.  The matrix kernels then add a bias with four
// 16-byte loads per 32 scores and lane: fp16 B21 S1512 H11 D72 with a [B,1,Sq,Sk] causal and
// padding mask, forward + backward 2.50 -> 1.37 ms.
__global__ __launch_bounds__(256) void bias_prepare_kernel(const AttnArgs a, int64_t heads,
                                                           int rows, int pitch,
                                                           float* __restrict__ out) {
    const int64_t quad = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int per_row = pitch / 4;
    const int64_t row = quad / per_row;
    const int x = (int)(quad - row * per_row) * 4;  // first slot
    const int64_t bh = row / rows;
    const int i = (int)(row - bh * rows);
    const int64_t b = bh / heads, h = bh - b * heads;
    if (b >= a.batch) return;
    const int g = (x >> 4) & 1, r = x & 15;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int j = (x & ~31) + acc_row(r + e, g);
        if (i < a.sq && j < a.sk)
            v[e] = bias_log2(bias_load(a, b * a.bs[0] + h * a.bs[1] + (int64_t)i * a.bs[2] +
                                              (int64_t)j * a.bs[3]));
    }
    *reinterpret_cast<f32x4_t*>(out + row * pitch + x) = v;
}

int64_t prepared_rows(int64_t n) { return (n + 63) & ~int64_t(63); }

bool half_ptrs_ok(std::initializer_list<const void*> ptrs) {
    for (const void* p : ptrs)
        if (!p || !aligned16(p)) return false;
    return true;
}

}  // namespace


extern "C" size_t slapo_amd_attn_keep_mask_bytes(const slapo_attn_params* p) {
    if (!p || !(p->p_drop > 0.f) || (p->dtype != SLAPO_F16 && p->dtype != SLAPO_BF16)) return 0;
    if (p->batch <= 0 || p->heads <= 0 || p->seqlen_q <= 0 || p->seqlen_k <= 0) return 0;
    const size_t words = (size_t)((p->seqlen_k + 31) / 32) * (size_t)((p->seqlen_q + 3) & ~3);
    return (size_t)p->batch * p->heads * words * sizeof(uint32_t);
}

namespace {

// One query per sequence without dropout: attn_decode.hip.  How many workgroups share the keys of one
// (batch, head), 0 where that kernel does not apply.
int decode_shares(const slapo_attn_params* p) {
    if (!p || p->seqlen_q != 1 || p->p_drop > 0.f || p->batch <= 0 || p->heads <= 0 ||
        p->seqlen_k <= 0)
        return 0;
    return attn_decode_shares((int64_t)p->batch * p->heads, p->causal ? 1 : p->seqlen_k);
}

}  // namespace

namespace {

BiasKind bias_kind(const slapo_attn_params* p, int bias_type) {
    if (bias_type == SLAPO_BIAS_NONE) return kNoBias;
    if (bias_type == SLAPO_BIAS_PREPARED) return kPreparedBias;
    return p->seqlen_q == 1 || p->bias_strides[2] == 0 ? kKeyBias : kScoreBias;
}
BiasKind bias_kind(const slapo_attn_params* p, const AttnArgs& a) {
    return bias_kind(p, a.has_bias ? a.bias_type : SLAPO_BIAS_NONE);
}

// Row blocks and tiles of a call, for the current device.
struct Extent {
    int64_t cus, blocks_q, blocks_k, tiles_q, tiles_k;
    bool f32, causal;
    explicit Extent(const slapo_attn_params* p) {
        cus = cus_of_current_device();
        f32 = p->dtype == SLAPO_F32;
        causal = p->causal && p->window <= 0;
        const int64_t n_bh = (int64_t)p->batch * p->heads, rows = f32 ? 64 : 128, tile = f32 ? 32 : 64;
        auto blocks = [&](int64_t n) { return n_bh * ((n + rows - 1) / rows); };
        auto tiles = [&](int64_t n) {
            return ((p->window > 0 && p->window + rows < n ? p->window + rows : n) + tile - 1) / tile;
        };
        blocks_q = blocks(p->seqlen_q), blocks_k = blocks(p->seqlen_k);
        tiles_q = tiles(p->seqlen_q), tiles_k = tiles(p->seqlen_k);
    }
    static bool known(const slapo_attn_params* p) {
        return p && p->batch > 0 && p->heads > 0 && p->seqlen_q > 0 && p->seqlen_k > 0 && p->head_dim > 0;
    }
};

// Into how many shares the forward of a call deals the tiles of a row block.
int plan_forward(const slapo_attn_params* p, BiasKind kind) {
    const Extent e(p);
    const int shares = attn_splits(e.blocks_q, e.cus, e.tiles_k, e.f32, e.causal);
    if (e.f32 || kind == kScoreBias) return shares;
    // Groups of wavefronts in a workgroup do the same without partial results in memory.  (Which dropout it is
    // matters to calls of few tiles only, which are not dealt.)
    const int groups = attn_fwd_groups(e.blocks_q, e.cus, e.tiles_k, p->head_dim, e.causal, kind,
                                       p->p_drop > 0.f ? 1 : 0);
    if (groups == 1 || shares > groups) return shares;
    // Dealt all the same, above head_dim 64: beyond 40 tiles, where the merge is the smaller part, and, above 96,
    // where two groups read a bias for one workgroup a CU (dealt / two groups: causal B1 S2048 H16 with a padding
    // mask 51.2 / 53.2 us, p 0.1 74.5 / 77.7, without a mask 56.1 / 47.5; H8 with a [B,1,Sq,Sk] mask 54.1 / 60.8, causal
    // 50.8 / 57.9, with p 0.1 both the same).
    if (p->head_dim > 64 && e.tiles_k > 40) return shares;
    const bool half = 2 * e.blocks_q <= e.cus;
    if (p->head_dim > 96 && groups == 2 &&
        (kind == kKeyBias ? !half : kind == kPreparedBias && half && !(p->p_drop > 0.f)))
        return shares;
    return 1;
}
size_t forward_bytes(const slapo_attn_params* p, BiasKind kind) {
    const size_t shares = plan_forward(p, kind);
    return shares == 1 ? 0
                       : shares * p->batch * p->heads * p->seqlen_q * (2 + p->head_dim) * sizeof(float);
}

// Whether a backward runs as one launch (attn_bwd_both_impl.h): while the workgroups of both kernels
// together are fewer than two such launches would keep resident.  Device time of the backward, two
// launches -> delta_kernel and one: bf16 B4 S512 H8 D64 (256 workgroups) 25.4 -> 18.6 us, B6 S1187 H4
// D64 causal (480) 48.5 -> 36.3, B2 S1024 H12 D80 causal (384) 61.9 -> 40.8, B8 S512 H12 D64 (768) 39.9
// -> 38.1; B8 S1024 H8 D64 (1024) 71.1 -> 69.7, D80 102 -> 104.  At head_dim 128 a CU holds one workgroup
// of dK/dV: B2 S1024 H12 causal (384) 75.8 -> 51.3, B2 S1024 H16 (512) 82.6 -> 80.9.
// With a prepared bias, forward and backward at bf16 B2 S1024 H12: D64 97.2 -> 85.0 us, causal 97.7 -> 81.9,
// D80 causal 140 -> 111, D128 causal 170 -> 108; with stored keep bits as well D128 202 -> 138, but at
// head_dim 81-96 the one kernel spills (174 -> 263).
bool one_launch_backward(const slapo_attn_params* p, const Extent& e, BiasKind kind, int dropout) {
    if (dropout != 0 && dropout != 3) return false;
    if (kind == kScoreBias) return false;
    if (kind == kPreparedBias && dropout && p->head_dim > 80 && p->head_dim <= 96) return false;
    return e.blocks_q + e.blocks_k < (p->head_dim <= 96 ? 4 : 2) * e.cus;
}

// Up to how many tiles per block the one launch also stands in for two shares.  Its two kernels fill each
// other's idle CUs and write no partial results, but it lasts as long as an undivided dK/dV block: what it
// saves (the partial results and their merge, 12 to 35 us) does not grow with the length, what it costs
// does, and more so where the blocks differ (keys that are padded) or a tile takes longer.  Where two of its
// workgroups share a CU, above half as many blocks as CUs, the line lies twice as far out, and farther where
// nearly all CUs have two.  Backward, two shares / one launch, bf16, B1:
//   S2048 H8 (128 blocks, 32 tiles)  D64 66.7 / 49.8 us, padded keys 64.4 / 52.3, [B,1,Sq,Sk] 82.9 / 76.8, p 0.1
//                                    72.2 / 58.6; D80 85.6 / 65.7; D128 109 / 83.1, padded keys 91.5 / 81.2
//   S4096 H4 (128, 64 tiles)         D64 99.2 / 86.0, all keys valid 1 / 0.89, padded 1 / 0.97 to 1, [B,1,Sq,Sk]
//                                    1 / 1.10; D80 134 / 123, padded 1 / 1.06; D128 166 / 149, padded 1 / 1.09,
//                                    [B,1,Sq,Sk] 1 / 0.87
//   S8192 H2 (128, 128 tiles)        D64 160 / 157, D80 236 / 239, D128 297 / 294; p 0.1 D64 1 / 1.06, D128 1 / 0.92;
//                                    padded 1 / 1.13 to 1.25
//   S16384 H1 (128, 256 tiles)       D32 1 / 0.96, D64 274 / 287, D80 406 / 428, D128 519 / 539; padded 1 / 1.22 to 1.38
//   causal, 192 blocks               S4096 H6 D64 105 / 89.1, padded 1 / 0.89; S8192 H3 171 / 163, padded 1 / 1.02
//   causal, 256 blocks               S2048 H16 D64 86.8 / 55.0, D80 110 / 74.4; S8192 H4 D64 217 / 175, padded 1 /
//                                    0.89, p 0.1 1 / 0.80, both 1 / 0.92
// With dropout at head_dim 65 to 96 the two kernels have builds of their own for few blocks, which the one launch
// has not: its line lies nearer (D80 causal, two shares / one launch: p 0.1 S3072 H7 (168 blocks) 1 / 0.95, H10
// (240) 1 / 0.83; with padded keys S2048 H12 (192) 1 / 0.92, S3072 H7 1 / 1.07; with a [B,1,Sq,Sk] mask S1536 H18
// (216) 1 / 0.88, S2048 H12 1 / 1.03).  In three and four shares, whose line would lie below 32 tiles, nothing is
// replaced: S2048 H5 (80 blocks) D64 48.5 / 46.2, D80 66.4 / 68.6; H4 (64) D64 49.5 / 45.6, D80 57.6 / 62.9, S4096 H2
// D64 62.3 / 78.6.
int one_launch_tiles(const slapo_attn_params* p, const Extent& e, BiasKind kind, int dropout) {
    // [head_dim][dropout][bias: none, per key, prepared][blocks: up to half of the CUs, 0.8, more]
    static constexpr int kTiles[4][2][3][3] = {
        {{{256, 384, 384}, {48, 96, 192}, {64, 80, 120}}, {{48, 96, 256}, {32, 64, 128}, {32, 64, 96}}},
        {{{128, 256, 384}, {64, 128, 192}, {40, 80, 120}}, {{64, 128, 192}, {40, 80, 128}, {32, 64, 96}}},
        {{{128, 256, 384}, {48, 96, 144}, {40, 80, 120}}, {{48, 48, 192}, {26, 32, 60}, {0, 24, 32}}},
        {{{128, 256, 384}, {48, 96, 144}, {96, 192, 288}}, {{128, 256, 384}, {48, 96, 144}, {40, 80, 120}}}};
    const int width = p->head_dim <= 32 ? 0 : p->head_dim <= 64 ? 1 : p->head_dim <= 96 ? 2 : 3;
    const int64_t blocks = (e.blocks_q + e.blocks_k) / 2;
    return kTiles[width][dropout != 0][kind][10 * blocks > 8 * e.cus ? 2 : 2 * blocks > e.cus ? 1 : 0];
}

// How a backward runs: in how many shares each kernel deals its tiles, or as one launch
// (attn_bwd_both_impl.h), which deals none.
struct BackwardPlan {
    int dq = 1, dkv = 1;
    bool one_launch = false;
};
// dropout: as in AttnArgs.  deal: whether there is room for partial results.
BackwardPlan plan_backward(const slapo_attn_params* p, BiasKind kind, int dropout, bool deal) {
    const Extent e(p);
    BackwardPlan plan;
    if (deal) {
        plan.dq = attn_splits(e.blocks_q, e.cus, e.tiles_k, e.f32, e.causal);
        plan.dkv = attn_splits(e.blocks_k, e.cus, e.tiles_q, e.f32, e.causal);
    }
    const int shares = std::max(plan.dq, plan.dkv);
    const int64_t tiles = std::max(e.tiles_q, e.tiles_k);
    if (!e.f32 && one_launch_backward(p, e, kind, dropout) &&
        (shares == 1 || (shares == 2 && tiles <= one_launch_tiles(p, e, kind, dropout)))) {
        plan.dq = plan.dkv = 1;
        plan.one_launch = true;
    }
    return plan;
}
size_t delta_bytes(const slapo_attn_params* p) {  // rounded: the partial results follow
    return (slapo_amd_attn_bwd_workspace_bytes(p) + 255) & ~size_t(255);
}
size_t backward_bytes(const slapo_attn_params* p, const BackwardPlan& plan) {
    if (plan.dq == 1 && plan.dkv == 1) return slapo_amd_attn_bwd_workspace_bytes(p);
    const size_t row = (size_t)p->batch * p->heads * p->head_dim * sizeof(float);
    return delta_bytes(p) + (plan.dq > 1 ? row * p->seqlen_q * plan.dq : 0) +
           (plan.dkv > 1 ? 2 * row * p->seqlen_k * plan.dkv : 0);
}

}  // namespace

extern "C" size_t slapo_amd_attn_fwd_workspace_bytes_for(const slapo_attn_params* prm, int bias_type) {
    if (!Extent::known(prm)) return 0;
    if (const int shares = decode_shares(prm))
        return shares == 1 ? 0
                           : (size_t)shares * prm->batch * prm->heads * (2 + prm->head_dim) *
                                 sizeof(float);
    return forward_bytes(prm, bias_kind(prm, bias_type));
}

extern "C" size_t slapo_amd_attn_bwd_ex_workspace_bytes_for(const slapo_attn_params* prm, int bias_type) {
    if (!Extent::known(prm)) return slapo_amd_attn_bwd_workspace_bytes(prm);
    const int dropout = !(prm->p_drop > 0.f) ? 0 : prm->keep_mask ? 3 : 1;
    return backward_bytes(prm, plan_backward(prm, bias_kind(prm, bias_type), dropout, true));
}

// Without the type: what is enough for every one of them.
extern "C" size_t slapo_amd_attn_fwd_workspace_bytes(const slapo_attn_params* prm) {
    size_t most = 0;
    for (int type : {SLAPO_BIAS_NONE, SLAPO_F32, SLAPO_BIAS_PREPARED})
        most = std::max(most, slapo_amd_attn_fwd_workspace_bytes_for(prm, type));
    return most;
}

extern "C" size_t slapo_amd_attn_bwd_ex_workspace_bytes(const slapo_attn_params* prm) {
    size_t most = 0;
    for (int type : {SLAPO_BIAS_NONE, SLAPO_F32, SLAPO_BIAS_PREPARED})
        most = std::max(most, slapo_amd_attn_bwd_ex_workspace_bytes_for(prm, type));
    return most;
}

extern "C" size_t slapo_amd_attn_prepared_bias_bytes(int64_t batch, int64_t heads,
                                                     int64_t seqlen_q, int64_t seqlen_k) {
    if (batch <= 0 || heads <= 0 || seqlen_q <= 0 || seqlen_k <= 0) return 0;
    // the kernels address the rows of one (batch, head) with 32-bit byte offsets
    const int64_t one = prepared_rows(seqlen_q) * prepared_rows(seqlen_k);
    if (one >= int64_t(1) << 30) return 0;
    return (size_t)(batch * heads * one) * sizeof(float);
}

extern "C" int slapo_amd_attn_prepare_bias(const void* bias, int bias_type,
                                           const int64_t bias_strides[4], int64_t batch,
                                           int64_t heads, int64_t seqlen_q, int64_t seqlen_k,
                                           float* out, void* stream) {
    if (!bias || !bias_strides || !out) return SLAPO_ERR_ARG;
    if (bias_type != SLAPO_F32 && bias_type != SLAPO_F16 && bias_type != SLAPO_BF16)
        return SLAPO_ERR_DTYPE;
    if (!aligned16(out)) return SLAPO_ERR_ALIGN;
    if (!slapo_amd_attn_prepared_bias_bytes(batch, heads, seqlen_q, seqlen_k))
        return SLAPO_ERR_SHAPE;
    AttnArgs a = {};
    a.bias = bias, a.bias_type = bias_type;
    for (int i = 0; i < 4; ++i) a.bs[i] = bias_strides[i];
    a.batch = (int)batch, a.sq = (int)seqlen_q, a.sk = (int)seqlen_k;
    const int rows = (int)prepared_rows(seqlen_q), pitch = (int)prepared_rows(seqlen_k);
    const int64_t quads = batch * heads * rows * (pitch / 4);
    const int64_t blocks = (quads + 255) / 256;
    if (blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    hipLaunchKernelGGL(bias_prepare_kernel, dim3((unsigned)blocks), dim3(256), 0,
                       (hipStream_t)stream, a, heads, rows, pitch, out);
    return check_launch();
}

extern "C" int slapo_amd_attn_fwd_ex(const slapo_attn_params* prm, const void* q, const void* k,
                                     const void* v, const void* bias, int bias_type, void* o,
                                     float* lse, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    AttnArgs a = {};
    int rc = fill_args(prm, &a, false);
    if (rc != SLAPO_OK) return rc;
    if (!q || !k || !v || !o || !lse) return SLAPO_ERR_ARG;
    if (workspace && !aligned16(workspace)) return SLAPO_ERR_ALIGN;
    a.q = q, a.k = k, a.v = v, a.o = o, a.lse = lse;
    const bool f32 = prm->dtype == SLAPO_F32;
    rc = set_bias(&a, bias, bias_type, f32, false);
    if (rc != SLAPO_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (!f32 && !half_ptrs_ok({q, k, v, o})) return SLAPO_ERR_ALIGN;
    if (int shares = decode_shares(prm)) {
        // 16-byte reads of whole rows (16-bit types: checked above)
        const bool rows_ok = !f32 || (a.d % 4 == 0 && strides_ok(prm->q_strides, 4) &&
                                      strides_ok(prm->k_strides, 4) &&
                                      strides_ok(prm->v_strides, 4) && half_ptrs_ok({q, k, v}));
        if (!workspace || workspace_bytes < slapo_amd_attn_fwd_workspace_bytes_for(prm, bias_type)) shares = 1;
        if (rows_ok && bias_type != SLAPO_BIAS_PREPARED)
            return attn_decode(a, prm->dtype, shares, static_cast<float*>(workspace), st);
    }
    if (workspace && decode_shares(prm) == 0) {
        const BiasKind kind = bias_kind(prm, a);
        if (workspace_bytes >= forward_bytes(prm, kind)) a.n_split = plan_forward(prm, kind);
        a.part = static_cast<float*>(workspace);
    }
    auto merged = [&](int status) {
        return status == SLAPO_OK && a.n_split > 1 ? attn_merge_fwd(a, prm->dtype, st) : status;
    };
    if (f32) return merged(attn_fwd_f32(a, st));
    if (a.dropout && a.keep_mask && (a.window > 0 || a.dropout == 2) && keep_mask_kernel_fits(a)) {
        // Local window, or a mask geometry without whole Philox blocks per aligned group of keys,
        // with a buffer for the keep bits: draw them first, the forward kernel then reads them
        // like the backward kernels do (bf16 B4 S2048 H16 D128, window 256, p 0.1: 88 against 127
        // us; the geometry: see keep_mask_kernel).  Otherwise the forward draws them itself and
        // stores them as it goes: there the Philox arithmetic overlaps the matrix instructions
        // and a separate pass measured slower (239 against 199 us at the same shape, 116
        // against 87 us at fp16 B8 S1024 H16 D64).
        rc = draw_keep_mask(a, st);
        if (rc != SLAPO_OK) return rc;
        a.dropout = 3;
    }
    return merged(prm->dtype == SLAPO_F16 ? attn_fwd_mfma_f16(a, st) : attn_fwd_mfma_bf16(a, st));
}

extern "C" int slapo_amd_attn_fwd(const slapo_attn_params* prm, const void* q, const void* k,
                                  const void* v, const float* bias, void* o, float* lse,
                                  void* stream) {
    return slapo_amd_attn_fwd_ex(prm, q, k, v, bias, SLAPO_F32, o, lse, nullptr, 0, stream);
}

extern "C" size_t slapo_amd_attn_bwd_workspace_bytes(const slapo_attn_params* prm) {
    if (!prm || prm->batch <= 0 || prm->heads <= 0 || prm->seqlen_q <= 0 || prm->head_dim <= 0)
        return 0;
    const size_t rows = (size_t)prm->batch * prm->heads * prm->seqlen_q;
    return rows * sizeof(float);  // delta
}

namespace {
int run_backward(const slapo_attn_params* prm, const void* q, const void* k, const void* v,
                 const void* bias, int bias_type, const void* o, const void* dout,
                 const float* lse, void* dq, void* dk, void* dv, const int64_t dq_strides[3],
                 const int64_t dk_strides[3], const int64_t dv_strides[3], void* workspace,
                 size_t workspace_bytes, int stages, bool deal, void* stream) {
    AttnArgs a = {};
    int rc = fill_args(prm, &a, true);
    if (rc != SLAPO_OK) return rc;
    if (!q || !k || !v || !o || !dout || !lse || !dq || !dk || !dv || !dq_strides ||
        !dk_strides || !dv_strides)
        return SLAPO_ERR_ARG;
    if (stages <= 0 || stages > SLAPO_BWD_ALL) return SLAPO_ERR_ARG;
    if (!workspace || workspace_bytes < slapo_amd_attn_bwd_workspace_bytes(prm) ||
        !aligned16(workspace))
        return SLAPO_ERR_WORKSPACE;
    for (int i = 0; i < 3; ++i) {
        a.dqs[i] = dq_strides[i];
        a.dks[i] = dk_strides[i];
        a.dvs[i] = dv_strides[i];
    }
    a.q = q, a.k = k, a.v = v, a.o = const_cast<void*>(o), a.dout = dout;
    a.lse = const_cast<float*>(lse);
    a.dk = dk, a.dv = dv;
    rc = set_bias(&a, bias, bias_type, prm->dtype == SLAPO_F32, true);
    if (rc != SLAPO_OK) return rc;
    hipStream_t st = (hipStream_t)stream;

    a.delta = reinterpret_cast<float*>(workspace);
    a.dq = dq;

    const bool f32 = prm->dtype == SLAPO_F32;
    if (!f32) {
        if (!half_ptrs_ok({q, k, v, o, dout, dq, dk, dv})) return SLAPO_ERR_ALIGN;
        if (!strides_ok(dq_strides, 8) || !strides_ok(dk_strides, 8) || !strides_ok(dv_strides, 8))
            return SLAPO_ERR_ALIGN;
    }
    // Partial results need room.  Both kernels' are merged in one launch at the end.
    BackwardPlan plan;
    float *dq_part = nullptr, *dkv_part = nullptr;
    if (deal) {
        const BiasKind kind = bias_kind(prm, a);
        plan = plan_backward(prm, kind, a.dropout, true);
        if (workspace_bytes < backward_bytes(prm, plan)) plan = plan_backward(prm, kind, a.dropout, false);
        float* next = reinterpret_cast<float*>(static_cast<char*>(workspace) + delta_bytes(prm));
        if (plan.dq > 1) {
            dq_part = next;
            next += (int64_t)plan.dq * a.batch * a.heads * a.sq * a.d;
        }
        if (plan.dkv > 1) dkv_part = next;
    }

    if (plan.one_launch)
        return prm->dtype == SLAPO_F16 ? attn_bwd_both_mfma_f16(a, st)
                                       : attn_bwd_both_mfma_bf16(a, st);
    // PREPARE has nothing to do (the dQ kernel computes delta for its own rows and stores it for
    // the dK / dV kernel), so DQ runs before DKDV.
    if (stages & SLAPO_BWD_DQ) {
        a.n_split = plan.dq, a.part = dq_part;
        rc = f32                        ? attn_bwd_dq_f32(a, st)
             : prm->dtype == SLAPO_F16 ? attn_bwd_dq_mfma_f16(a, st)
                                       : attn_bwd_dq_mfma_bf16(a, st);
        if (rc != SLAPO_OK) return rc;
    }
    if (stages & SLAPO_BWD_DKDV) {
        a.n_split = plan.dkv, a.part = dkv_part;
        rc = f32                        ? attn_bwd_f32(a, st)
             : prm->dtype == SLAPO_F16 ? attn_bwd_mfma_f16(a, st)
                                       : attn_bwd_mfma_bf16(a, st);
        if (rc != SLAPO_OK) return rc;
    }
    return dq_part || dkv_part
               ? attn_merge_bwd(a, prm->dtype, dq_part, plan.dq, dkv_part, plan.dkv, st)
               : SLAPO_OK;
}

}  // namespace

extern "C" int slapo_amd_attn_bwd_stages(const slapo_attn_params* prm, const void* q,
                                         const void* k, const void* v, const float* bias,
                                         const void* o, const void* dout, const float* lse,
                                         void* dq, void* dk, void* dv,
                                         const int64_t dq_strides[3], const int64_t dk_strides[3],
                                         const int64_t dv_strides[3], void* workspace,
                                         size_t workspace_bytes, int stages, void* stream) {
    return run_backward(prm, q, k, v, bias, SLAPO_F32, o, dout, lse, dq, dk, dv, dq_strides,
                        dk_strides, dv_strides, workspace, workspace_bytes, stages, false, stream);
}

extern "C" int slapo_amd_attn_bwd_ex(const slapo_attn_params* prm, const void* q, const void* k,
                                     const void* v, const void* bias, int bias_type,
                                     const void* o, const void* dout, const float* lse, void* dq,
                                     void* dk, void* dv, const int64_t dq_strides[3],
                                     const int64_t dk_strides[3], const int64_t dv_strides[3],
                                     void* workspace, size_t workspace_bytes, void* stream) {
    return run_backward(prm, q, k, v, bias, bias_type, o, dout, lse, dq, dk, dv, dq_strides,
                        dk_strides, dv_strides, workspace, workspace_bytes, SLAPO_BWD_ALL, true,
                        stream);
}

extern "C" int slapo_amd_attn_bwd(const slapo_attn_params* prm, const void* q, const void* k,
                                  const void* v, const float* bias, const void* o,
                                  const void* dout, const float* lse, void* dq, void* dk,
                                  void* dv, const int64_t dq_strides[3],
                                  const int64_t dk_strides[3], const int64_t dv_strides[3],
                                  void* workspace, size_t workspace_bytes, void* stream) {
    return slapo_amd_attn_bwd_stages(prm, q, k, v, bias, o, dout, lse, dq, dk, dv, dq_strides,
                                     dk_strides, dv_strides, workspace, workspace_bytes,
                                     SLAPO_BWD_ALL, stream);
}

// ---- backward without a caller workspace -------------------------------------------------------
// delta = rowsum(dO * O) lives in an array of the library's own, so that callers that must not
// allocate (HIP graph capture, serving loops) need no workspace: every device that runs the
// library holds one copy of the array until the process ends.
namespace {

constexpr size_t kScratchFloats = size_t(1) << 20;  // 4 MiB: batch * heads * seqlen_q <= 1 048 576
__device__ __align__(256) float scratch[kScratchFloats];

std::mutex scratch_lock;
float* scratch_of_device[64] = {};  // device address of `scratch`, per device, once resolved

// The array's name is only a handle on the host; its address on the current device comes from
// the runtime, once per device.
int scratch_on_current_device(float** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return SLAPO_ERR_DEVICE;
    std::lock_guard<std::mutex> guard(scratch_lock);
    if (!scratch_of_device[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
            return SLAPO_ERR_DEVICE;
        scratch_of_device[dev] = static_cast<float*>(p);
    }
    *out = scratch_of_device[dev];
    return SLAPO_OK;
}

}  // namespace

extern "C" int slapo_amd_attn_bwd_static_scratch(
    const slapo_attn_params* prm, const void* q, const void* k, const void* v, const float* bias,
    const void* o, const void* dout, const float* lse, void* dq, void* dk, void* dv,
    const int64_t dq_strides[3], const int64_t dk_strides[3], const int64_t dv_strides[3],
    void* stream) {
    const size_t need = slapo_amd_attn_bwd_workspace_bytes(prm);
    if (need == 0) return SLAPO_ERR_SHAPE;
    if (need > kScratchFloats * sizeof(float)) return SLAPO_ERR_WORKSPACE;
    float* ws = nullptr;
    const int rc = scratch_on_current_device(&ws);
    if (rc != SLAPO_OK) return rc;
    return slapo_amd_attn_bwd_stages(prm, q, k, v, bias, o, dout, lse, dq, dk, dv, dq_strides,
                                     dk_strides, dv_strides, ws, kScratchFloats * sizeof(float),
                                     SLAPO_BWD_ALL, stream);
}
