// FusedQKV's re-layout (slapo/op/linear.py:41-57): the projection's columns are [heads, head_size, 3],
// q, k and v of one element side by side; attention wants three dense [.., heads, head_size] tensors.
// Forward: one read of the packed rows, one write of each of the three; backward: the other way
// round.  torch takes three strided copies forward and, backward, three zero-filled packed tensors
// and their sum.  Bound by memory: 2 x the packed bytes.  A thread owns V consecutive elements of
// each of q, k, v = 3 V consecutive packed elements: 16-byte accesses on both sides.
// fp16 tokens 8192, hidden 1024 (100 MB): 16.1 us, 6.2 TB/s; forward + backward 122 -> 54 us.
#include "common.h"

using namespace slapo;

namespace {

template <typename T, int V>
struct alignas(V == 1 ? sizeof(T) : 16) Run {
    T v[V];
};

template <typename T, int V, bool kJoin>
__global__ __launch_bounds__(256) void qkv_kernel(T* __restrict__ packed, T* __restrict__ q,
                                                  T* __restrict__ k, T* __restrict__ v,
                                                  int64_t n_runs) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= n_runs) return;
    typedef Run<T, V> run_t;
    T* const dst[3] = {q, k, v};
    run_t wide[3], one[3];
    if constexpr (kJoin) {
#pragma unroll
        for (int i = 0; i < 3; ++i) one[i] = *reinterpret_cast<const run_t*>(dst[i] + c * V);
#pragma unroll
        for (int e = 0; e < 3 * V; ++e) wide[e / V].v[e % V] = one[e % 3].v[e / 3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
            *reinterpret_cast<run_t*>(packed + (3 * c + i) * V) = wide[i];
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i)
            wide[i] = *reinterpret_cast<const run_t*>(packed + (3 * c + i) * V);
#pragma unroll
        for (int e = 0; e < 3 * V; ++e) one[e % 3].v[e / 3] = wide[e / V].v[e % V];
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<run_t*>(dst[i] + c * V) = one[i];
    }
}

// Elements are moved, not computed with: 2- and 4-byte types stand for all.
template <typename T, bool kJoin>
int launch(void* packed, void* q, void* k, void* v, int64_t n, hipStream_t st) {
    constexpr int V = 16 / sizeof(T);
    const bool vec = n % V == 0 && aligned16(packed) && aligned16(q) && aligned16(k) && aligned16(v);
    const int64_t runs = vec ? n / V : n;
    const int64_t blocks = (runs + 255) / 256;
    if (blocks > 0x7FFFFFFF) return SLAPO_ERR_SHAPE;
    if (vec)
        hipLaunchKernelGGL((qkv_kernel<T, V, kJoin>), dim3((unsigned)blocks), dim3(256), 0, st,
                           (T*)packed, (T*)q, (T*)k, (T*)v, runs);
    else
        hipLaunchKernelGGL((qkv_kernel<T, 1, kJoin>), dim3((unsigned)blocks), dim3(256), 0, st,
                           (T*)packed, (T*)q, (T*)k, (T*)v, runs);
    return check_launch();
}

template <bool kJoin>
int run(void* packed, void* q, void* k, void* v, int64_t n, int dtype, void* stream) {
    if (!packed || !q || !k || !v) return SLAPO_ERR_ARG;
    if (n <= 0) return SLAPO_ERR_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case SLAPO_F32: return launch<uint32_t, kJoin>(packed, q, k, v, n, st);
        case SLAPO_F16:
        case SLAPO_BF16: return launch<uint16_t, kJoin>(packed, q, k, v, n, st);
        default: return SLAPO_ERR_DTYPE;
    }
}

}  // namespace

extern "C" int slapo_amd_qkv_split(const void* packed, void* q, void* k, void* v, int64_t n,
                                   int dtype, void* stream) {
    return run<false>(const_cast<void*>(packed), q, k, v, n, dtype, stream);
}

extern "C" int slapo_amd_qkv_join(const void* q, const void* k, const void* v, void* packed,
                                  int64_t n, int dtype, void* stream) {
    return run<true>(packed, const_cast<void*>(q), const_cast<void*>(k), const_cast<void*>(v), n,
                     dtype, stream);
}
