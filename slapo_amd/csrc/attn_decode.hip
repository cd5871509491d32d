// Attention of ONE query per sequence against its keys (a generation step): forward only, no
// dropout.  There is nothing to multiply in tiles here -- a key costs 4 D operations for 4 D bytes of
// fp16 / bf16 -- so the kernel is bound by reading K and V once, and what the tile kernel
// (attn_fwd_impl.h, 128 query rows per workgroup) lacks is workgroups: batch * heads of them, each
// walking all keys in turn.
//
// A workgroup takes one (batch, head) and a contiguous share of its keys; the share is dealt to the
// four wavefronts in strips.  16 bytes per lane: a row of D elements is read by the kLanes lanes of a
// power of two that covers it, so a wavefront has 64 / kLanes keys per load and kStrip loads of K
// and of V in flight.  Each row group of a wavefront keeps its own running maximum, sum and output;
// groups, then wavefronts, are merged once at the end.  With more than one share per (batch, head)
// the unnormalised results go to a workspace and attn_decode_merge_kernel adds them in order (no
// atomics).  Scores, probabilities and sums are fp32; q, k, v enter as they are stored.
// bf16 B8 H16 Sk2000 D128 (131 MB): 54.6 us with the tile kernel, 27.5 us here (4.8 TB/s).
//
// Reference semantics: slapo/op/attention.py:163-181 (attention_bmk).
#include <type_traits>

#include "attn_common.h"

using namespace slapo;

namespace {

constexpr int kThreads = 256;
constexpr int kStrip = 4;  // keys per row group and round trip

template <typename T>
struct Row16 {  // 16 bytes of a row
    static constexpr int kN = Elem<T>::kPerVec;
    T v[kN];
};

// sum_e q[e] k[e], products exact, fp32 sums
template <typename T>
__device__ __forceinline__ float dot16(const Row16<T>& q, const Row16<T>& k) {
    float s = 0.f;
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_fmaf(q.v[e], k.v[e], s);
    } else {
        typedef T pair_t __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const pair_t a = {q.v[e], q.v[e + 1]}, b = {k.v[e], k.v[e + 1]};
            if constexpr (std::is_same<T, f16_t>::value)
                s = __builtin_amdgcn_fdot2(a, b, s, false);
            else
                s = __builtin_amdgcn_fdot2_f32_bf16(a, b, s, false);
        }
    }
    return s;
}

// Sum over the kLanes lanes of a row group, on each of them: DPP moves inside a 16-lane row (quad
// permutes, then mirrors of 8 and of 16), no LDS traffic.
template <int kCtrl>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), kCtrl, 0xF, 0xF, false));
}
template <int kLanes>
__device__ __forceinline__ float lanes_sum(float v) {
    static_assert(kLanes == 4 || kLanes == 8 || kLanes == 16 || kLanes == 32, "");
    v += dpp_move<0xB1>(v);                           // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);                           // quad_perm [2,3,0,1]
    if constexpr (kLanes >= 8) v += dpp_move<0x141>(v);   // row_half_mirror
    if constexpr (kLanes >= 16) v += dpp_move<0x140>(v);  // row_mirror
    if constexpr (kLanes >= 32) v += __shfl_xor(v, 16, 64);
    return v;
}

// Scores are kept in natural units for fp32 (accurate expf) and in log2 units otherwise.
template <typename T>
constexpr bool kLog2Units = sizeof(T) != 4;
template <typename T>
__device__ __forceinline__ float exp_units(float x) {
    if constexpr (kLog2Units<T>)
        return fast_exp2(x);
    else
        return expf(x);
}

// One merge of (m, l, o) states: m is -inf where nothing has been seen.
template <typename T>
__device__ __forceinline__ float weight_of(float m, float m_all) {
    return m == -INFINITY ? 0.f : exp_units<T>(m - m_all);
}

// Partial results of one share, fp32: [share][batch * heads][2 + d] = m, l, o (unnormalised).
template <typename T>
__device__ __forceinline__ void finish_row(const AttnArgs& a, int bh, float m, float l, float o,
                                           int c) {
    const int b = bh / a.heads, h = bh % a.heads;
    T* out = reinterpret_cast<T*>(a.o) + b * a.os[0] + h * a.os[2];
    out[c] = Elem<T>::from_f32(o * (1.0f / l));
    if (c == 0) {
        const float unit = kLog2Units<T> ? kLn2 : 1.0f;
        // a row that saw nothing but masked keys: see canonical_bias
        const float log_l = kLog2Units<T> ? __builtin_log2f(l) : logf(l);
        a.lse[bh] = m == -kFltMax ? l * kMaskedRowLse : (m + log_l) * unit;
    }
}

template <typename T, int kLanes>
__global__ __launch_bounds__(kThreads) void attn_decode_kernel(const AttnArgs a, int share_keys,
                                                               float* __restrict__ part) {
    constexpr int kN = Row16<T>::kN;
    constexpr int kGroups = 64 / kLanes;     // keys per wavefront and load
    constexpr int kSpan = kGroups * kStrip;  // keys per wavefront and round trip
    __shared__ float sh_m[4], sh_l[4];
    __shared__ float sh_o[4][kLanes * kN];
    const int n_bh = a.batch * a.heads;
    const int bh = blockIdx.x % n_bh, share = blockIdx.x / n_bh;
    const int b = bh / a.heads, h = bh % a.heads;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane % kLanes, group = lane / kLanes;
    const int n_keys = a.causal ? 1 : a.sk;  // the query is row 0: a causal mask leaves key 0
    const int k_lo = share * share_keys;
    int k_hi = min(k_lo + share_keys, n_keys);

    const T* qp = reinterpret_cast<const T*>(a.q) + b * a.qs[0] + h * a.qs[2];
    const T* kp = reinterpret_cast<const T*>(a.k) + b * a.ks[0] + h * a.ks[2];
    const T* vp = reinterpret_cast<const T*>(a.v) + b * a.vs[0] + h * a.vs[2];
    const bool bias = a.has_bias != 0;
    const int64_t bias_at = b * a.bs[0] + h * a.bs[1];
    const bool col_ok = sub * kN < a.d;
    const int col = min(sub * kN, a.d - kN);

    if (bias && bias_load(a, bias_at) > kMaskedBias) {
        // Padding at the end of the share contributes exactly zero to a row that sees key 0 (see
        // key_bias_span): its keys are not read.
        int last = k_lo - 1;
        for (int j = k_lo + (int)threadIdx.x; j < k_hi; j += kThreads)
            if (bias_load(a, bias_at + (int64_t)j * a.bs[3]) > kMaskedBias) last = j;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) last = max(last, __shfl_xor(last, off, 64));
        if (lane == 0) sh_m[wave] = __int_as_float(last);
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 4; ++w) last = max(last, __float_as_int(sh_m[w]));
        k_hi = last + 1;
        __syncthreads();
    }

    Row16<T> q = {};
    if (col_ok) *reinterpret_cast<u32x4_t*>(&q) = *reinterpret_cast<const u32x4_t*>(qp + col);
    const float scale = kLog2Units<T> ? a.scale_log2 : a.scale;

    float m = -INFINITY, l = 0.f, o[kN];
#pragma unroll
    for (int e = 0; e < kN; ++e) o[e] = 0.f;
    for (int j0 = k_lo + wave * kSpan; j0 < k_hi; j0 += 4 * kSpan) {
        Row16<T> kk[kStrip], vv[kStrip];
        float s[kStrip];
#pragma unroll
        for (int u = 0; u < kStrip; ++u) {
            const int64_t j = min(j0 + u * kGroups + group, k_hi - 1);
            *reinterpret_cast<u32x4_t*>(&kk[u]) =
                __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(kp + j * a.ks[1] + col));
            *reinterpret_cast<u32x4_t*>(&vv[u]) =
                __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vp + j * a.vs[1] + col));
            s[u] = bias ? bias_load(a, bias_at + j * a.bs[3]) : 0.f;
        }
        if (j0 + kSpan > k_hi) {  // rows past the end: zeros, as 0 * inf would not be one
#pragma unroll
            for (int u = 0; u < kStrip; ++u)
                if (j0 + u * kGroups + group >= k_hi) vv[u] = Row16<T>{};
        }
        float mx = m;
#pragma unroll
        for (int u = 0; u < kStrip; ++u) {
            float t = dot16<T>(q, kk[u]);  // (q is zero past the last column)
            t = lanes_sum<kLanes>(t) * scale;
            if (bias) t += kLog2Units<T> ? bias_log2(s[u]) : canonical_bias(s[u]);
            s[u] = j0 + u * kGroups + group < k_hi ? t : -INFINITY;
            mx = fmaxf(mx, s[u]);
        }
        const float alpha = weight_of<T>(m, mx);
        const float ref = mx == -INFINITY ? 0.f : mx;
        m = mx;
        l *= alpha;
#pragma unroll
        for (int e = 0; e < kN; ++e) o[e] *= alpha;
#pragma unroll
        for (int u = 0; u < kStrip; ++u) {
            const float p = exp_units<T>(s[u] - ref);
            l += p;
#pragma unroll
            for (int e = 0; e < kN; ++e)
                o[e] = __builtin_fmaf(p, Elem<T>::to_f32(vv[u].v[e]), o[e]);
        }
    }
    // row groups of the wavefront
#pragma unroll
    for (int off = kLanes; off < 64; off <<= 1) {
        const float m2 = __shfl_xor(m, off, 64), l2 = __shfl_xor(l, off, 64);
        const float mx = fmaxf(m, m2);
        const float w1 = weight_of<T>(m, mx), w2 = weight_of<T>(m2, mx);
        m = mx;
        l = l * w1 + l2 * w2;
#pragma unroll
        for (int e = 0; e < kN; ++e) o[e] = o[e] * w1 + __shfl_xor(o[e], off, 64) * w2;
    }
    // wavefronts
    if (lane == 0) sh_m[wave] = m, sh_l[wave] = l;
    if (group == 0) {
#pragma unroll
        for (int e = 0; e < kN; ++e) sh_o[wave][sub * kN + e] = o[e];
    }
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= a.d) return;
    const float m_all = fmaxf(fmaxf(sh_m[0], sh_m[1]), fmaxf(sh_m[2], sh_m[3]));
    float l_all = 0.f, o_all = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const float wt = weight_of<T>(sh_m[w], m_all);
        l_all = __builtin_fmaf(sh_l[w], wt, l_all);
        o_all = __builtin_fmaf(sh_o[w][c], wt, o_all);
    }
    if (!part) {
        finish_row<T>(a, bh, m_all, l_all, o_all, c);
    } else {
        float* p = part + ((int64_t)share * n_bh + bh) * (2 + a.d);
        if (c == 0) p[0] = m_all, p[1] = l_all;
        p[2 + c] = o_all;
    }
}

template <typename T>
__global__ __launch_bounds__(128) void attn_decode_merge_kernel(const AttnArgs a, int n_shares,
                                                                const float* __restrict__ part) {
    const int n_bh = a.batch * a.heads;
    const int bh = blockIdx.x, c = threadIdx.x;
    if (c >= a.d) return;
    const int64_t step = (int64_t)n_bh * (2 + a.d);
    const float* p = part + (int64_t)bh * (2 + a.d);
    float m = -INFINITY, l = 0.f, o = 0.f;
    for (int s0 = 0; s0 < n_shares; s0 += 8) {  // eight shares requested together
        float ms[8], ls[8], os[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float* r = p + min(s0 + u, n_shares - 1) * step;
            ms[u] = r[0], ls[u] = r[1], os[u] = r[2 + c];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (s0 + u >= n_shares) break;
            const float mx = fmaxf(m, ms[u]);
            const float w1 = weight_of<T>(m, mx), w2 = weight_of<T>(ms[u], mx);
            m = mx;
            l = l * w1 + ls[u] * w2;
            o = o * w1 + os[u] * w2;
        }
    }
    finish_row<T>(a, bh, m, l, o, c);
}

template <typename T, int kLanes>
int launch(const AttnArgs& a, int n_shares, int share_keys, float* part, hipStream_t st) {
    const int64_t n_bh = (int64_t)a.batch * a.heads;
    const int64_t blocks = n_bh * n_shares;
    if (blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    hipLaunchKernelGGL((attn_decode_kernel<T, kLanes>), dim3((unsigned)blocks), dim3(kThreads), 0,
                       st, a, share_keys, n_shares > 1 ? part : nullptr);
    int rc = check_launch();
    if (rc != SLAPO_OK || n_shares == 1) return rc;
    hipLaunchKernelGGL(attn_decode_merge_kernel<T>, dim3((unsigned)n_bh), dim3(128), 0, st, a,
                       n_shares, (const float*)part);
    return check_launch();
}

template <typename T>
int dispatch(const AttnArgs& a, int n_shares, int share_keys, float* part, hipStream_t st) {
    const int lanes = (a.d + Elem<T>::kPerVec - 1) / Elem<T>::kPerVec;
    if (lanes <= 4) return launch<T, 4>(a, n_shares, share_keys, part, st);
    if (lanes <= 8) return launch<T, 8>(a, n_shares, share_keys, part, st);
    if (lanes <= 16) return launch<T, 16>(a, n_shares, share_keys, part, st);
    return launch<T, 32>(a, n_shares, share_keys, part, st);
}

}  // namespace

namespace slapo {

// Shares of the keys: enough workgroups for four per CU (1024 on 256 CUs), none with fewer than 128
// keys (two round trips per wavefront at head_dim 128; less does not pay for the merge).
int attn_decode_shares(int64_t n_bh, int n_keys) {
    const int64_t want = (1024 + n_bh - 1) / n_bh, most = (n_keys + 127) / 128;
    return (int)(want < most ? want : most);
}

int attn_decode(const AttnArgs& a, int dtype, int n_shares, float* part, hipStream_t st) {
    const int n_keys = a.causal ? 1 : a.sk;
    const int share_keys = (n_keys + n_shares - 1) / n_shares;
    switch (dtype) {
        case SLAPO_F32: return dispatch<float>(a, n_shares, share_keys, part, st);
        case SLAPO_F16: return dispatch<f16_t>(a, n_shares, share_keys, part, st);
        default: return dispatch<bf16_t>(a, n_shares, share_keys, part, st);
    }
}

}  // namespace slapo
