// Philox4x32-10 counter-based RNG and the element -> (subsequence, counter, lane) mapping that
// ATen's fused dropout kernels use, written once for host and device so the two agree bit for
// bit.  The mapping (reference call sites: torch.nn.functional.dropout at
// slapo/op/fused_bias.py:74 and slapo/op/attention.py:179-180):
//
//   launch:  block = 256 threads, grid = min(num_cus * (max_threads_per_cu / 256),
//            ceil(numel / 256)), T = 256 * grid subsequences, one per thread;
//   vector kernel (vec in {2,4,8,16}): thread t, loop trip m handles the `vec` consecutive
//            elements starting at (m * T + t) * vec and draws ceil(vec/4) Philox blocks per
//            trip; element e of the group uses word e % 4 of block e / 4;
//   scalar kernel (vec == 1): thread t, loop trip m draws one block; word w belongs to
//            element t + T * (4 * m + w);
//   Philox block number c of subsequence t under generator state (seed, offset) has
//            key = seed, counter = { lo(offset/4 + c), hi(offset/4 + c), lo(t), hi(t) };
//   keep iff  2^-32 + float(word) * 2^-32 < float(1 - p)   (rocRAND's uniform conversion).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define SLAPO_HD __host__ __device__ __forceinline__
#else
#define SLAPO_HD inline
#endif

namespace slapo {

struct u32x4 {
    uint32_t x, y, z, w;
};

// a ^ b ^ c.  On the device one instruction (v_bitop3_b32 with the truth table of a three-way XOR)
// where two v_xor_b32 would be needed: a Philox round is then two multiplications and two of
// these instead of two and four.
SLAPO_HD uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
#else
    return a ^ b ^ c;
#endif
}

SLAPO_HD u32x4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                             uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c1, k0);
        const uint32_t n1 = (uint32_t)p1;
        const uint32_t n2 = xor3((uint32_t)(p0 >> 32), c3, k1);
        const uint32_t n3 = (uint32_t)p0;
        c0 = n0;
        c1 = n1;
        c2 = n2;
        c3 = n3;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return u32x4{c0, c1, c2, c3};
}

// Everything a kernel needs to regenerate mask bits; filled on the host.
struct DropoutState {
    uint32_t key0, key1;      // seed lo / hi
    uint64_t base_counter;    // offset / 4
    uint64_t total_threads;   // T
    uint32_t vec;             // 1,2,4,8,16
    uint32_t calls_per_iter;  // ceil(vec/4), 1 for vec==1
    uint32_t keep_max;        // keep iff word <= keep_max (unless keep_none)
    uint32_t keep_none;       // 1: nothing is kept (p == 1)
    int32_t t_shift;          // log2(T) when T is a power of two, else -1
    int32_t g_shift;          // log2(vec / 4) when vec >= 4, else -1
    float inv_keep;           // 1 / (1 - p)
    // NULL, or device memory holding {seed, offset}: a kernel then takes key and base counter
    // from there (resolve_device_state) instead of the three fields above
    const uint64_t* device_state;
};

#if defined(__HIPCC__)
// First statement of every kernel that draws: a uniform branch and one 16-byte uniform read.
__device__ __forceinline__ void resolve_device_state(DropoutState& s) {
    if (s.device_state != nullptr) {
        const uint64_t seed = s.device_state[0];
        const uint64_t offset = s.device_state[1];
        s.key0 = (uint32_t)seed;
        s.key1 = (uint32_t)(seed >> 32);
        s.base_counter = offset >> 2;
    }
}
#endif

SLAPO_HD void split_by_threads(const DropoutState& s, uint64_t v, uint64_t& thread,
                               uint64_t& trip) {
    if (s.t_shift >= 0) {
        trip = v >> s.t_shift;
        thread = v & (s.total_threads - 1);
    } else {
        trip = v / s.total_threads;
        thread = v - trip * s.total_threads;
    }
}

SLAPO_HD u32x4 philox_block(const DropoutState& s, uint64_t thread, uint64_t call) {
    const uint64_t c = s.base_counter + call;
    return philox4x32_10((uint32_t)c, (uint32_t)(c >> 32), (uint32_t)thread,
                         (uint32_t)(thread >> 32), s.key0, s.key1);
}

SLAPO_HD bool keep_word(const DropoutState& s, uint32_t w) {
    return (w <= s.keep_max) && !s.keep_none;
}

// Keep-bit of one element (any vec).  Costs a full Philox block per element.
SLAPO_HD bool dropout_keep1(const DropoutState& s, uint64_t elem) {
    uint64_t thread, trip, call;
    uint32_t lane;
    if (s.vec == 1) {
        uint64_t q;
        split_by_threads(s, elem, thread, q);
        call = q >> 2;
        lane = (uint32_t)(q & 3);
    } else {
        const uint64_t v = elem / s.vec;
        const uint32_t e = (uint32_t)(elem - v * s.vec);
        split_by_threads(s, v, thread, trip);
        call = trip * s.calls_per_iter + (e >> 2);
        lane = e & 3;
    }
    const u32x4 r = philox_block(s, thread, call);
    const uint32_t w = lane == 0 ? r.x : lane == 1 ? r.y : lane == 2 ? r.z : r.w;
    return keep_word(s, w);
}

// Keep-bits (bit i <-> element 4*group + i) of an aligned group of four consecutive elements.
// Valid only when vec is 4, 8 or 16 (one Philox block covers the group).
SLAPO_HD uint32_t dropout_keep4(const DropoutState& s, uint64_t group) {
    const uint32_t groups_per_vec = s.vec >> 2;  // 1, 2 or 4
    uint64_t v, sub;
    if (groups_per_vec == 1) {
        v = group;
        sub = 0;
    } else if (groups_per_vec == 2) {
        v = group >> 1;
        sub = group & 1;
    } else {
        v = group >> 2;
        sub = group & 3;
    }
    uint64_t thread, trip;
    split_by_threads(s, v, thread, trip);
    const u32x4 r = philox_block(s, thread, trip * s.calls_per_iter + sub);
    return (keep_word(s, r.x) ? 1u : 0u) | (keep_word(s, r.y) ? 2u : 0u) |
           (keep_word(s, r.z) ? 4u : 0u) | (keep_word(s, r.w) ? 8u : 0u);
}

// dropout_keep4 for the common launch geometry: vec >= 4 and a power-of-two thread count, so the
// element -> (subsequence, counter) split is shifts and masks only.
SLAPO_HD uint32_t dropout_keep4_pow2(const DropoutState& s, uint64_t group) {
    const uint64_t v = group >> s.g_shift;
    const uint32_t sub = (uint32_t)group & ((1u << s.g_shift) - 1u);
    const uint64_t thread = v & (s.total_threads - 1);
    const uint64_t trip = v >> s.t_shift;
    const u32x4 r = philox_block(s, thread, trip * s.calls_per_iter + sub);
    return (keep_word(s, r.x) ? 1u : 0u) | (keep_word(s, r.y) ? 2u : 0u) |
           (keep_word(s, r.z) ? 4u : 0u) | (keep_word(s, r.w) ? 8u : 0u);
}

// What the first three rounds of the blocks of one counter share.  Counter word 0 and 1 (offset / 4 +
// call) are the same for all subsequences of a call and word 3 is zero below 2^32 subsequences, so
// that one of the two products of round 1 and one of round 2 belong to the call: a block takes 18
// multiplications and 18 XORs instead of 20 and 20, and no 64-bit index arithmetic: 47 vector
// instructions with its keep bits (push_keep4), 61 to 74 before.  Forward with dropout in the kernel and
// backward, fp16 B8 S1024 H16 D64 causal: 162 -> 155 us, bf16 B4 S2048 H16 D128 causal 451 -> 436;
// keep_mask_kernel at window 256 of that shape 23.5 -> 20.4.
struct PhiloxCall {
    uint32_t a, b, c, d;
    uint32_t key0, key1;
};
SLAPO_HD PhiloxCall philox_call(uint64_t counter, uint32_t key0, uint32_t key1) {
    const uint32_t c0 = (uint32_t)counter, c1 = (uint32_t)(counter >> 32);
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;                     // round 1
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * ((uint32_t)(p0 >> 32) ^ key1);  // round 2
    return {c1 ^ key0, (uint32_t)(p1 >> 32) ^ (key0 + 0x9E3779B9u),
            (uint32_t)p0 ^ (key1 + 0xBB67AE85u), (uint32_t)p1 ^ (key0 + 2u * 0x9E3779B9u), key0,
            key1};
}
SLAPO_HD u32x4 philox_block(const PhiloxCall& s, uint32_t thread) {
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * thread;                 // round 1
    const uint64_t p0 = (uint64_t)0xD2511F53u * ((uint32_t)(p1 >> 32) ^ s.a);  // round 2
    const uint64_t q0 = (uint64_t)0xD2511F53u * ((uint32_t)p1 ^ s.b);   // round 3
    const uint64_t q1 = (uint64_t)0xCD9E8D57u * ((uint32_t)(p0 >> 32) ^ s.c);
    uint32_t k0 = s.key0 + 2u * 0x9E3779B9u, k1 = s.key1 + 2u * 0xBB67AE85u;
    uint32_t c0 = (uint32_t)(q1 >> 32) ^ s.d, c1 = (uint32_t)q1;
    uint32_t c2 = xor3((uint32_t)(q0 >> 32), (uint32_t)p0, k1), c3 = (uint32_t)q0;
#pragma unroll
    for (int r = 3; r < 10; ++r) {
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
        const uint64_t m0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t m1 = (uint64_t)0xCD9E8D57u * c2;
        c0 = xor3((uint32_t)(m1 >> 32), c1, k0);
        c1 = (uint32_t)m1;
        c2 = xor3((uint32_t)(m0 >> 32), c3, k1);
        c3 = (uint32_t)m0;
    }
    return u32x4{c0, c1, c2, c3};
}
// `bits` shifted up by the block's four keep bits (bit i <-> word i): two instructions a word, a
// compare and an addition with its carry.
SLAPO_HD uint32_t push_keep4(uint32_t bits, const u32x4& r, uint32_t keep_max) {
    bits = bits + bits + (r.w <= keep_max ? 1u : 0u);
    bits = bits + bits + (r.z <= keep_max ? 1u : 0u);
    bits = bits + bits + (r.y <= keep_max ? 1u : 0u);
    return bits + bits + (r.x <= keep_max ? 1u : 0u);
}
// Does PhiloxCall serve this plan?  One block per group of four elements and trip (the plan of a 4-byte
// tensor), 32-bit subsequences.
SLAPO_HD bool philox_call_fits(const DropoutState& s) {
    return s.vec == 4 && (s.total_threads >> 32) == 0 && !s.keep_none;
}

// Keep-bits of the n (1..32) consecutive elements starting at elem, for any launch geometry and
// alignment.  Deliberately a rolled loop: this path is rare and must stay small.
SLAPO_HD uint32_t dropout_keep_any(const DropoutState& s, uint64_t elem, int n) {
    uint32_t bits = 0;
#if defined(__HIPCC__)
#pragma unroll 1
#endif
    for (int e = 0; e < n; ++e) bits |= (dropout_keep1(s, elem + (uint64_t)e) ? 1u : 0u) << e;
    return bits;
}

// Keep-bits of the kN (a multiple of four, at most 32) consecutive elements starting at elem (bit j <->
// element elem + j), for any launch geometry and alignment.  The split of the element index, a division
// where the thread count is no power of two, is taken once.  From vec 4 on kN / 4 + 1 blocks are drawn
// (kAligned, elem % 4 == 0: one fewer), at vec 2 kN / 2 + 1, at vec 1 kN.
template <int kN, bool kAligned = false>
SLAPO_HD uint32_t dropout_keep_run(const DropoutState& s, uint64_t elem) {
    const uint64_t v = elem >> __builtin_ctz(s.vec);
    uint64_t thread, trip;
    if (((v | s.total_threads) >> 32) == 0 && s.t_shift < 0) {
        trip = (uint32_t)v / (uint32_t)s.total_threads;
        thread = (uint32_t)v - (uint32_t)trip * (uint32_t)s.total_threads;
    } else {
        split_by_threads(s, v, thread, trip);
    }
    constexpr int kBlocks = kN / 4 + (kAligned ? 0 : 1);
    bool one_call = philox_call_fits(s) && thread + kBlocks <= s.total_threads;
#if defined(__HIP_DEVICE_COMPILE__)
    one_call = __builtin_amdgcn_ballot_w64(!one_call) == 0;
#endif
    uint64_t all = 0;
    if (one_call) {
        const PhiloxCall call = philox_call(s.base_counter + trip, s.key0, s.key1);
        const uint32_t t = (uint32_t)thread;
        uint32_t last = 0, bits = 0;
        if constexpr (!kAligned)
            last = push_keep4(0u, philox_block(call, t + kN / 4), s.keep_max);
#pragma unroll
        for (int blk = kN / 4 - 1; blk >= 0; --blk)
            bits = push_keep4(bits, philox_block(call, t + blk), s.keep_max);
        all = (((uint64_t)last << kN) | bits) >> (kAligned ? 0 : elem & 3u);
    } else {  // other words a block or blocks a trip, or a run that wraps to the next call
        const int step = s.vec < 4 ? (int)s.vec : 4;  // elements a block serves
        const int skip = (int)elem & (step - 1);      // ... of the first one before elem
        uint32_t sub = (uint32_t)(elem >> 2) & (s.calls_per_iter - 1u), run = 0;
#if defined(__HIPCC__)
#pragma unroll 1
#endif
        for (int at = -skip; at < kN; at += step) {
            const u32x4 r =
                philox_block(s, thread, s.vec == 1 ? trip >> 2 : trip * s.calls_per_iter + sub);
            uint32_t four = s.keep_none ? 0u : push_keep4(0u, r, s.keep_max);
            if (step == 1) four = (four >> (trip & 3)) & 1u;
            if (step == 2) four &= 3u;
            run |= at < 0 ? four >> -at : four << at;
            if (++sub < s.calls_per_iter) continue;
            sub = 0;
            if (++thread == s.total_threads) thread = 0, ++trip;
        }
        all = run;
    }
    return (uint32_t)all & (kN == 32 ? ~0u : (1u << (kN & 31)) - 1u);
}

}  // namespace slapo
