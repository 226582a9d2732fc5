// zh_sample.hip -- the output shortlist of stochastic decoding: the top-k
// logits (k <= 64), highest first, ties to the lower token id, as the
// reference's GPU session hands them to its CPU sampler
// (Session.runOutputShortlist, runtime/gpu/session.zig:789-828; topk_f32,
// matvec.metal:1568-1651; sampleShortlist, sampling.zig:31-45).
//
// Two launches over packed keys (ordered value bits << 32 | ~id, so the
// largest key is the largest value and, among equal values, the lowest id):
//   partial  workgroup b takes logits [4096 b, 4096 b + 4096) and leaves its
//            k largest keys, in any order;
//   final    one workgroup, every partial workgroup's k keys: the top k, as
//            entries in order.
// Both select by wavefront (16 keys a lane, then the four wavefronts' 4k
// candidates): the k-th largest is found bit by bit from the top, each bit one
// count of the keys at or above it by ballots, so the cost does not grow with
// k; the order of the final k is each key's count of larger ones.  128256
// logits: 40 of them in 13.9 + 9.7 us, where k rounds of a wavefront
// maximum took 31.4 + 53.2 us.
#include "zh_internal.h"

namespace zh {

constexpr int kSlice = 4096;         // logits per partial workgroup
constexpr int kShortMax = 64;        // longest shortlist (max_shortlist_len, runtime/gpu/types.zig:119)
__device__ __forceinline__ unsigned long long short_key(float v, uint32_t id) {
    const uint32_t b = __float_as_uint(v);
    const uint32_t o = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return ((unsigned long long)o << 32) | (unsigned long long)(0xFFFFFFFFu - id);
}

// The largest t > 0 that at least k of the wavefront's N x 64 items reach (0 if none): at(i, c) says
// whether item i of this lane reaches c.
template <int N, class At> __device__ __forceinline__ uint32_t wave_kth(int k, At at) {
    uint32_t t = 0;
#pragma unroll 1
    for (uint32_t bit = 0x80000000u; bit; bit >>= 1) {
        const uint32_t c = t | bit;
        int n = 0;
#pragma unroll
        for (int i = 0; i < N; i++) n += __popcll(__ballot(at(i, c)));
        if (n >= k) t = c;
        if (n == k) break;
    }
    return t;
}
// The wavefront's k largest keys (all of them if fewer are not 0) into dst[0 .. k), the rest of dst 0.
template <int N>
__device__ __forceinline__ void wave_select(const unsigned long long (&key)[N], int k, unsigned long long *dst) {
    const int lane = threadIdx.x & 63;
    uint32_t hi[N], lo[N];
#pragma unroll
    for (int i = 0; i < N; i++) hi[i] = (uint32_t)(key[i] >> 32), lo[i] = (uint32_t)key[i];
    const uint32_t t = wave_kth<N>(k, [&](int i, uint32_t c) { return hi[i] >= c; });
    int above = 0, equal = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        above += __popcll(__ballot(hi[i] > t));
        equal += __popcll(__ballot(hi[i] == t && lo[i]));
    }
    // more keys of the k-th value than places: the largest low words, i.e. the lowest ids (the
    // low word of a key is 0 for no id below 2^32 - 1: an empty place)
    const uint32_t l =
        above + equal > k ? wave_kth<N>(k - above, [&](int i, uint32_t c) { return hi[i] == t && lo[i] >= c; }) : 1u;
    int base = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const bool take = hi[i] > t || (hi[i] == t && lo[i] >= l);
        const unsigned long long m = __ballot(take);
        if (take) dst[base + __popcll(m & ((1ull << lane) - 1ull))] = key[i];
        base += __popcll(m);
    }
    if (lane >= base && lane < k) dst[lane] = 0ull;
}

// The workgroup's k largest of its four wavefronts' keys, into dst in any order (wavefront 0 writes).
__device__ __forceinline__ void group_select(const unsigned long long (&key)[16], int k, unsigned long long *dst) {
    __shared__ unsigned long long cand[4][kShortMax];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    wave_select<16>(key, k, cand[wave]);
    __syncthreads();
    if (wave == 0) {
        unsigned long long c[4];
#pragma unroll
        for (int i = 0; i < 4; i++) c[i] = lane < k ? cand[i][lane] : 0ull;
        wave_select<4>(c, k, dst);
    }
}

__global__ void __launch_bounds__(256) shortlist_partial_kernel(const float *__restrict__ x, int n, int k,
                                                                unsigned long long *__restrict__ keys) {
    const int base = blockIdx.x * kSlice + threadIdx.x;
    unsigned long long key[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int idx = base + 256 * i;
        key[i] = idx < n ? short_key(x[min(idx, n - 1)], (uint32_t)idx) : 0ull;
    }
    group_select(key, k, keys + (size_t)blockIdx.x * k);
}

__global__ void __launch_bounds__(256) shortlist_final_kernel(const unsigned long long *__restrict__ keys, int nkeys,
                                                              int k, uint32_t *__restrict__ entries) {
    __shared__ unsigned long long top[kShortMax];
    unsigned long long key[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int j = threadIdx.x + 256 * i;
        key[i] = j < nkeys ? keys[min(j, nkeys - 1)] : 0ull;
    }
    group_select(key, k, top);
    __syncthreads();
    if ((int)threadIdx.x < k) {
        const unsigned long long v = top[threadIdx.x];
        int r = 0;
        for (int j = 0; j < k; j++) r += top[j] > v;
        // entry r: {u32 token id, f32 logit} (ShortlistEntry, runtime/gpu/types.zig:114-117)
        const uint32_t o = (uint32_t)(v >> 32);
        const uint32_t bits = (o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o;
        entries[2 * r] = 0xFFFFFFFFu - (uint32_t)(v & 0xFFFFFFFFull);
        entries[2 * r + 1] = bits;
    }
}

size_t shortlist_scratch_keys(int n) { return (size_t)((n + kSlice - 1) / kSlice) * kShortMax; }

hipError_t launch_shortlist(const float *x, int n, int k, unsigned long long *keys, uint32_t *entries,
                            hipStream_t s) {
    const int blocks = (n + kSlice - 1) / kSlice;
    if (n < 1 || k < 1 || k > kShortMax || k > n || blocks * k > kSlice)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(shortlist_partial_kernel, dim3(blocks), dim3(256), 0, s, x, n, k, keys);
    hipLaunchKernelGGL(shortlist_final_kernel, dim3(1), dim3(256), 0, s, keys, blocks * k, k, entries);
    return hipGetLastError();
}

}  // namespace zh
