// The whole backward of a small attention call in one launch: the workgroups of the dK/dV kernel and,
// after them, those of the dQ kernel.  A kernel whose workgroups do not fill the chip ends with the
// longest of them, and two such kernels in a row take the sum; workgroups of both on a CU at a time
// fill each other's waits.  delta = rowsum(dO * O), which the dQ kernel otherwise hands on to the dK/dV
// kernel, comes from a small kernel ahead of them.
// Reference semantics: autograd of slapo/op/attention.py:163-181.
#pragma once
#include "attn_bwd_dq_impl.h"
#include "attn_bwd_impl.h"

namespace slapo {
namespace bwd_both {

// delta of every row, times the factor that the dK / dV kernel wants on it (lse_row_factor), in the order
// of dq_block's own sum, so that both give the same bits (rows that saw only masked keys aside: dq_block
// divides their factor out again, equal within a rounding): two lanes a row, lane g on columns 16 t + 8 g.
// Heads are the fastest index, as in memory.  Bound by reading dO and O once.
template <typename T, int kSteps, bool kBias>
__global__ __launch_bounds__(256) void delta_kernel(const AttnArgs a, int64_t n_rows) {
    const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / 2;
    const int g = (int)threadIdx.x & 1;
    const int64_t r = row < n_rows ? row : n_rows - 1;
    const int64_t bi = r / a.heads, h = r - bi * a.heads, b = bi / a.sq, i = bi - b * a.sq;
    const int64_t at = b * a.os[0] + i * a.os[1] + h * a.os[2];
    typedef typename Mma<T>::frag frag_t;
    u32x4_t gv[kSteps], ov[kSteps];
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
        const int col = min(16 * t + 8 * g, a.d - 8);
        gv[t] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(a.dout) + at + col);
        ov[t] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const T*>(a.o) + at + col);
    }
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
        const frag_t gf = __builtin_bit_cast(frag_t, keep_or_zero(gv[t], 16 * t + 8 * g < a.d));
        const frag_t of = __builtin_bit_cast(frag_t, ov[t]);
#pragma unroll
        for (int e = 0; e < 8; ++e) sum = __builtin_fmaf((float)gf[e], (float)of[e], sum);
    }
    sum += __shfl_xor(sum, 1, 64);
    if (g == 0 && row < n_rows) {
        const int64_t out = (b * a.heads + h) * a.sq + i;
        a.delta[out] = kBias ? sum * lse_row_factor(a.lse[out]) : sum;
    }
}

template <typename T, int DPAD, int kBias, int kDrop, int kSteps>
__global__ __launch_bounds__(256, bwd::bwd_per_cu(DPAD)) void attn_bwd_both_kernel(
    const AttnArgs dkv, const AttnArgs dq, int n_dkv) {
    const int block = (int)blockIdx.x;
    if (block < n_dkv)
        bwd::dkv_block<T, DPAD, kBias, kDrop, 1, kSteps, bwd::bwd_per_cu(DPAD), false>(dkv, block, n_dkv);
    else
        bwd_dq::dq_block<T, DPAD, kBias, kDrop, kSteps, false>(dq, block - n_dkv,
                                                               (int)gridDim.x - n_dkv);
}

template <typename T, int DPAD, int kBias, int kDrop, int kSteps>
int launch(const AttnArgs& a, hipStream_t st) {
    const int64_t n_bh = (int64_t)a.batch * a.heads;
    const int64_t n_dkv = (a.sk + 127) / 128 * n_bh, n_dq = (a.sq + 127) / 128 * n_bh;
    const int64_t n_rows = n_bh * a.sq;
    const int64_t delta_blocks = (n_rows * 2 + 255) / 256;
    if (n_dkv + n_dq > 0x7FFFFFFF || delta_blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    const size_t lds_dkv = bwd::BwdSmem<T, DPAD, false>::kBytes, lds_dq = bwd_dq::lds_bytes<T, DPAD, kBias>();
    const size_t smem = lds_dkv > lds_dq ? lds_dkv : lds_dq;
    auto kern = attn_bwd_both_kernel<T, DPAD, kBias, kDrop, kSteps>;
    static std::atomic<uint64_t> lds_ready{0};  // per instantiation, one bit per device
    if (allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, lds_ready) != SLAPO_OK)
        return SLAPO_ERR_LAUNCH;
    AttnArgs dkv = a, dq = a;
    set_dispatch_order(&dkv, n_dkv, bwd::bwd_per_cu(DPAD));
    set_dispatch_order(&dq, n_dq, bwd::bwd_per_cu(DPAD));
    hipLaunchKernelGGL((delta_kernel<T, kSteps, kBias != 0>), dim3((unsigned)delta_blocks), dim3(256), 0,
                       st, a, n_rows);
    if (const int rc = check_launch(); rc != SLAPO_OK) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(n_dkv + n_dq)), dim3(256), smem, st, dkv, dq, (int)n_dkv);
    return check_launch();
}

template <typename T, int DPAD, int kSteps = DPAD / 16>
int dispatch_flags(const AttnArgs& a, hipStream_t st) {
    if (!a.has_bias)
        return a.dropout ? launch<T, DPAD, 0, 3, kSteps>(a, st) : launch<T, DPAD, 0, 0, kSteps>(a, st);
    if (a.bias_type == SLAPO_BIAS_PREPARED) {
        if (!a.dropout) return launch<T, DPAD, 3, 0, kSteps>(a, st);
        if constexpr (kSteps != 6) return launch<T, DPAD, 3, 3, kSteps>(a, st);
        return SLAPO_ERR_SHAPE;  // (one_launch_backward)
    }
    return a.dropout ? launch<T, DPAD, 2, 3, kSteps>(a, st) : launch<T, DPAD, 2, 0, kSteps>(a, st);
}
// Calls without bias, with one value per key or with a prepared bias, without dropout or with stored bits.
template <typename T>
int dispatch(const AttnArgs& a, hipStream_t st) {
    if (a.d <= 32) return dispatch_flags<T, 32>(a, st);
    if (a.d <= 64) return dispatch_flags<T, 64>(a, st);
    if (a.d <= 80) return dispatch_flags<T, 96, 5>(a, st);
    if (a.d <= 96) return dispatch_flags<T, 96>(a, st);
    return dispatch_flags<T, 128>(a, st);
}

}  // namespace bwd_both
}  // namespace slapo
