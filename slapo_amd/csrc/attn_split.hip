// Merging the partial results of attention calls whose rows were walked by several workgroups.
//
// A call with few (batch, head) pairs and long sequences leaves most of the chip idle and takes as
// long as one workgroup needs for all its tiles.  The kernels then deal the tiles of a workgroup's
// rows to `n_split` workgroups (AttnArgs), each of which leaves an fp32 partial result in the
// caller's workspace: the forward (m, l, unnormalised O), the backward kernels plain partial sums.
// These kernels add them in a fixed order -- no atomics, bitwise reproducible -- reading every
// partial value once: bound by memory, n_split * 4 bytes per value.
#include <type_traits>

#include "attn_common.h"

using namespace slapo;

namespace {

constexpr int kThreads = 256;

template <typename T>
__device__ __forceinline__ void store4(T* p, const f32x4_t& v) {
    if constexpr (sizeof(T) == 4) {
        // (rows of fp32 tensors need no alignment)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[e] = v[e];
    } else {
        u32x2_t w;
        w.x = pack2<T>(v[0], v[1]), w.y = pack2<T>(v[2], v[3]);
        *reinterpret_cast<u32x2_t*>(p) = w;
    }
}

// Forward: a thread owns four columns of one query row.  m in log2 units.
template <typename T>
__global__ __launch_bounds__(kThreads) void merge_fwd_kernel(const AttnArgs a) {
    const int quads = (a.d + 3) / 4;
    const int64_t n_rows = (int64_t)a.batch * a.heads * a.sq;
    const int64_t at = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    const int64_t row = at / quads;
    if (row >= n_rows) return;
    const int c = (int)(at - row * quads) * 4;
    const int64_t plane = n_rows * a.d;
    const float* ml = a.part + a.n_split * plane + 2 * row;
    float m = -INFINITY;
    for (int s = 0; s < a.n_split; ++s) m = fmaxf(m, ml[2 * s * n_rows]);
    float l = 0.f;
    f32x4_t o = {0.f, 0.f, 0.f, 0.f};
    const int n = min(4, a.d - c);
    for (int s = 0; s < a.n_split; ++s) {
        const float ms = ml[2 * s * n_rows];
        // (no maximum: nothing seen, or nothing but NaN scores, whose sum and values are NaN and stay)
        const float w = ms == -INFINITY ? 0.f : fast_exp2(ms - m);
        l = __builtin_fmaf(ml[2 * s * n_rows + 1], w, l);
        const float* p = a.part + s * plane + row * a.d + c;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < n) o[e] = __builtin_fmaf(p[e], w, o[e]);
    }
    // the 16-bit kernels leave the factor of the kept probabilities to the output rows
    constexpr bool kF32 = sizeof(T) == 4;
    const float inv = (!kF32 && a.dropout ? a.rng.inv_keep : 1.0f) / l;
    const int i = (int)(row % a.sq);
    const int64_t bh = row / a.sq, b = bh / a.heads, h = bh - b * a.heads;
    T* out = reinterpret_cast<T*>(a.o) + b * a.os[0] + (int64_t)i * a.os[1] + h * a.os[2] + c;
    if (n == 4) {
        store4<T>(out, o * inv);
    } else {
        for (int e = 0; e < n; ++e) out[e] = Elem<T>::from_f32(o[e] * inv);
    }
    if (c == 0) {
        const float lse = kF32 ? row_lse(m, l) : (m + __builtin_log2f(l)) * kLn2;
        a.lse[row] = m == -kFltMax ? l * kMaskedRowLse : lse;
    }
}

// Backward: up to three tensors [batch, rows, heads, d], each the sum of n partial ones.
struct SumJob {
    const float* part;
    void* dst;
    int64_t strides[3];
    int rows, n;
    int64_t first;  // of the launch's threads
};
struct SumJobs {
    SumJob job[3];
    int count;
    int64_t total;
    int n_bh, heads, d;
};

template <typename T>
__global__ __launch_bounds__(kThreads) void merge_bwd_kernel(const SumJobs js) {
    const int64_t at = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (at >= js.total) return;
    int which = 0;
    while (which + 1 < js.count && at >= js.job[which + 1].first) ++which;
    const SumJob& j = js.job[which];
    const int quads = (js.d + 3) / 4;
    const int64_t local = at - j.first;
    const int64_t row = local / quads;
    const int c = (int)(local - row * quads) * 4;
    const int64_t plane = (int64_t)js.n_bh * j.rows * js.d;
    const float* p = j.part + row * js.d + c;
    const int n = min(4, js.d - c);
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < j.n; ++s, p += plane) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < n) v[e] += p[e];
    }
    const int64_t bh = row / j.rows, i = row - bh * j.rows;
    const int64_t b = bh / js.heads, h = bh - b * js.heads;
    T* out = reinterpret_cast<T*>(j.dst) + b * j.strides[0] + i * j.strides[1] + h * j.strides[2] + c;
    if (n == 4) {
        store4<T>(out, v);
    } else {
        for (int e = 0; e < n; ++e) out[e] = Elem<T>::from_f32(v[e]);
    }
}

template <typename F>
int by_type(int dtype, F&& f) {
    if (dtype == SLAPO_F32) return f(float());
    if (dtype == SLAPO_F16) return f(f16_t());
    return f(bf16_t());
}

}  // namespace

namespace slapo {

// Into how many workgroups the tiles of one row block are dealt: as many as the device has room for
// (`slots`), eight at most, none with fewer than six tiles (four of the slower fp32 ones) and none at
// all below 24 (12) tiles: partial results and their merging cost about 10 us, a tile of 64 keys
// takes a workgroup about 0.6 us at head_dim 64 and 1.1 us at 128.  1: no split.
// A CU is busy with one workgroup of the 16-bit kernels (one wavefront per SIMD does 92 % of what
// two do), with two of the fp32 ones.  Kernels, merging included, bf16, causal: B1 S2304 H3 D128
// forward 49 -> 29 us, forward + backward 206 -> 109 us; at B2 S1024 H8 D64 the same split costs
// (forward 19 -> 26 us).  fp32 B1 S1971 H2 D72 forward + backward 629 -> 170 us.
// Under a causal mask the blocks have half the longest one's tiles on average, so that even a launch
// with a workgroup for every CU gains from two shares (bf16 B1 S8192 H4 D128 backward 457 -> 339 us; where
// groups of wavefronts or the one-launch backward apply they take the place of two, attn_capi.hip).
int attn_splits(int64_t blocks, int64_t cus, int64_t tiles, bool f32, bool causal) {
    const int64_t slots = f32 ? 2 * cus : cus, least = f32 ? 4 : 6;
    if (blocks <= 0 || tiles < (f32 ? 12 : 24)) return 1;
    int64_t n = slots / blocks;
    if (n == 1 && causal) n = 2;
    if (n > tiles / least) n = tiles / least;
    if (n > 8) n = 8;
    return n < 2 ? 1 : (int)n;
}

// Into how many groups of wavefronts a forward workgroup of the 16-bit kernels is divided (attn_fwd_impl.h),
// for `blocks` undivided workgroups of 128 queries: four, two or one, so that their number comes near what
// the chip holds.  Four groups of a wavefront each bring the 32-query workgroups to four times as many; above
// head_dim 64 their LDS leaves one a CU.  Under a causal mask the workgroups have half the longest one's
// tiles on average, so more of them pay.  Forward, undivided (or by attn_splits) / two / four groups, bf16
// without a mask:
//   D64   B1 S1024 H4 (32 blocks) 17.8 / 12.1 / 9.7 us, H16 (128) 18.3 / 13.1 / 14.6, causal 18.3 / 13.0 /
//         11.1, H32 (256) 20.1 / 18.5 / 25.1, causal 19.4 / 13.8 / 19.1; B4 S512 H16 (256) 11.8 / 11.9 /
//         17.6, causal 11.9 / 9.3 / 15.5; B1 S8192 H4 causal (256) 93.8 / 72.6 / 68.1; with drawn dropout B1
//         S1024 H16 causal 39.3 / 24.1 / 16.5
//   D80   B1 S512 H16 (64) 13.6 / 11.8 / 12.5, S1024 H8 (64) 22.7 / 18.0 / 17.6, H16 (128) 23.4 / 19.1 /
//         32.5, H32 (256) 25.5 / 27.0 / 62.6, causal 24.2 / 20.5 / 48.7
//   D128  B1 S256 H16 (32) 9.9 / 10.4 / 9.9, S1024 H8 (64) 26.2 / 23.2 / 18.8, H16 (128) 27.2 / 24.9 / 34.8,
//         H32 causal (256) 27.7 / 31.7 / 49.8, S2048 H16 causal (256) 56.1 / 47.5 / 68.1
// Below six tiles there is nothing to divide (B1 S256 H16 D64 7.2 / 7.0 / 6.8).
// A prepared bias is read from memory by every workgroup, a second one per CU only where the chip has room:
// without drawn dropout two groups lose where it has little (undivided / two groups: D64 B1 S1024 H32 23.8 / 27.2,
// S8192 H4 197 / 227; D96 causal B4 S512 H16 17.8 / 22.1, B3 S777 H12 24.8 / 27.1, but B1 S1472 H16 (192 blocks)
// 37.9 / 31.6).  A padding mask leaves fewer tiles than the keys have (D128 B1 S512 H8, five of eight tiles valid,
// 12.6 / 13.6 / 13.5); drawing keep bits is worth dividing all the same (there 21.0 / - / 15.6).
int attn_fwd_groups(int64_t blocks, int64_t cus, int64_t tiles, int64_t d, bool causal, BiasKind bias,
                    int dropout) {
    if (cus <= 0 || blocks > cus || tiles < 6) return 1;
    const bool half = 2 * blocks <= cus, quarter = 4 * blocks <= cus;
    const bool rows = bias == kPreparedBias, drawn = dropout == 1 || dropout == 2;
    if (d <= 64) {
        if (quarter || (half && causal)) return 4;
        if (rows && !dropout && !half && !causal) return 1;
        return half || causal || tiles >= 16 ? 2 : 1;
    }
    if (d <= 96) {
        if (quarter && tiles >= 16) return 4;
        if (rows && !drawn && 4 * blocks > 3 * cus && tiles + (dropout != 0) <= 16)
            return 1;
        return half || causal ? 2 : 1;
    }
    if (quarter) return tiles >= (bias == kKeyBias && !drawn ? 12 : 8) ? 4 : 1;
    return tiles >= (half ? 8 : 24) && (half || causal) ? 2 : 1;
}

int attn_merge_fwd(const AttnArgs& a, int dtype, hipStream_t st) {
    const int64_t threads = (int64_t)a.batch * a.heads * a.sq * ((a.d + 3) / 4);
    const int64_t blocks = (threads + kThreads - 1) / kThreads;
    if (blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    return by_type(dtype, [&](auto t) {
        hipLaunchKernelGGL(merge_fwd_kernel<decltype(t)>, dim3((unsigned)blocks), dim3(kThreads), 0,
                           st, a);
        return check_launch();
    });
}

// dq_part / dkv_part: nullptr where that kernel was not split
int attn_merge_bwd(const AttnArgs& a, int dtype, const float* dq_part, int n_dq,
                   const float* dkv_part, int n_dkv, hipStream_t st) {
    SumJobs js = {};
    js.n_bh = a.batch * a.heads, js.heads = a.heads, js.d = a.d;
    const int64_t per_row = (a.d + 3) / 4;
    auto add = [&](const float* part, void* dst, const int64_t (&s)[3], int rows, int n) {
        SumJob& j = js.job[js.count++];
        j.part = part, j.dst = dst, j.rows = rows, j.n = n, j.first = js.total;
        for (int i = 0; i < 3; ++i) j.strides[i] = s[i];
        js.total += (int64_t)js.n_bh * rows * per_row;
    };
    if (dq_part) add(dq_part, a.dq, a.dqs, a.sq, n_dq);
    if (dkv_part) {
        add(dkv_part, a.dk, a.dks, a.sk, n_dkv);
        add(dkv_part + (int64_t)n_dkv * js.n_bh * a.sk * a.d, a.dv, a.dvs, a.sk, n_dkv);
    }
    if (!js.count) return SLAPO_OK;
    const int64_t blocks = (js.total + kThreads - 1) / kThreads;
    if (blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    return by_type(dtype, [&](auto t) {
        hipLaunchKernelGGL(merge_bwd_kernel<decltype(t)>, dim3((unsigned)blocks), dim3(kThreads), 0,
                           st, js);
        return check_launch();
    });
}

}  // namespace slapo
