// zh_pattn.hip -- causal attention of a prompt pass: many queries over the paged binary16 cache.
//
// A workgroup takes 128 (query, head) rows of one kv head -- 128 / G consecutive queries with its G
// query heads -- so every K/V tile read serves them all; a wavefront holds 32 rows.  Positions go in
// tiles of 64, one page each, two in LDS: K rows by the asynchronous copy, V through registers,
// transposed on the way (4 positions x 8 dims per thread), so that both products read their operand
// in one piece.  Workgroups with the most positions start first; kv heads alternate over the XCDs.
//
// S[position][row] = K Q^T on 32x32x16 products, Q as two binary16 pieces (K is exact): a lane then
// holds 16 positions of one row, so maximum, weights and sum stay in the lane (one exchange with
// the lane 32 on per tile), and O[dim][row] = V^T P^T takes the weights as they lie, in two pieces.
// The order of a product's reduction index is free as long as both operands share it: the weights'
// own.  Weights and sums are binary32.  The pieces are of the weights times 2^14 (outputs and sums
// carry the factor, which their quotient drops): both rounded to nearest, they hold a weight to 2^-22
// of itself, or to 2^-39 of the row's largest, so that thousands of small weights beside one large
// keep their sum.
//
// What bounds it: per tile and wavefront 64 matrix products (2048 cycles) and about 300 vector
// instructions (1200), two wavefronts per SIMD; 16384 queries x 32 heads over 16384 positions (head
// size 128) take 4.1 ms a layer (4.3 on another card), 1080 TFLOP/s of issued matrix work (the
// library's f16 product reaches 1180-1230 on the same card); the kernel before it, whose workgroups
// took four queries each and read the range again for every four, 15 ms.  Scaling the weights' pieces
// as it does costs 0.7% (1074 -> 1081 us over four passes of a layer), scaling the weights 5%.
//
// Few queries over many positions leave CUs idle: their positions are split over up to 16
// workgroups and a second launch merges.  (20 / 64 / 256 / 600 queries after 4000 positions, one
// layer of two: 540 / 564 / 810 / 1405 us a pass; unsplit 652 / 675 / 917 / 1427; the kernel
// before it 534 / 573 / 889 / 1608.)
#include <type_traits>

#include "zh_internal.h"

namespace zh {

typedef _Float16 ph2 __attribute__((ext_vector_type(2)));
typedef _Float16 ph4 __attribute__((ext_vector_type(4)));
typedef _Float16 ph8 __attribute__((ext_vector_type(8)));
typedef float pf16 __attribute__((ext_vector_type(16)));

constexpr int kPaRows = 128;  // query x head rows of a workgroup, 32 per wavefront
constexpr float kPaWeight = 16384.f;  // of the largest weight: its pieces below binary16's 65504

struct PAttnParams {
    const float *q;
    float *out;
    const __half *kc, *vc;
    const uint32_t *pages;
    int M, pos, G, nkv, kv_dim, q_stride, out_stride, qn;  // qn: queries per workgroup
    float qscale;                                          // score scale x log2 e
    // positions split over gridDim.y workgroups: their unnormalised outputs at part + z M heads HD
    // (row (query, head)), then {m, l} pairs at part_ml + z M heads 2
    float *part, *part_ml;
};

// of this lane and the one 32 apart
__device__ __forceinline__ float pair_max(float v) {
    uint32_t a, b;
    lane_pair<32>(__float_as_uint(v), a, b);
    return fmaxf(__uint_as_float(a), __uint_as_float(b));
}
__device__ __forceinline__ float pair_sum(float v) {
    uint32_t a, b;
    lane_pair<32>(__float_as_uint(v), a, b);
    return __uint_as_float(a) + __uint_as_float(b);
}

template <int HD> __global__ void __launch_bounds__(256, 2) pattn_kernel(PAttnParams p) {
    constexpr int KT = HD / 16, DT = HD / 32, C = HD / 8;  // 16-value steps, 32-dim tiles, 16-byte chunks of a row
    constexpr int KU = 64 * C / 256;                       // K chunks per thread and tile
    __shared__ __align__(16) uint4 ks0[64 * C], ks1[64 * C];          // K rows, chunks exchanged within a row
    __shared__ __align__(16) uint2 vs0[HD * 16], vs1[HD * 16];        // V transposed: 4 positions per word pair
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
    const int kvh = blockIdx.x % p.nkv, nqb = (p.M + p.qn - 1) / p.qn, qb = nqb - 1 - (int)blockIdx.x / p.nkv;
    const int q0 = qb * p.qn, qend = min(q0 + p.qn, p.M);
    const int kv_last = p.pos + qend - 1, nt_all = (kv_last >> 6) + 1;
    // this workgroup's tiles of 64 positions (one page each)
    const int ks = gridDim.y, z = blockIdx.y, t_begin = (int)((long long)z * nt_all / ks), nt = (int)((long long)(z + 1) * nt_all / ks);
    const int v = wave * 32 + l32, qi = q0 + v / p.G, head = kvh * p.G + v % p.G;
    const bool valid = v < p.qn * p.G && qi < p.M;
    const int qc = min(qi, qend - 1), qpos = p.pos + qc;
    const int wave_first = p.pos + min(q0 + wave * 32 / p.G, qend - 1);  // the wavefront's earliest query

    // the chunk that slot c of K row `row` holds
    auto swz = [](int row, int c) { return HD == 128 ? c ^ (row & 15) : HD == 64 ? c ^ ((row >> 1) & 7) : c; };
    auto vslot = [](int dim, int g) { return dim * 16 + (g ^ (((dim >> 1) & 15) ^ ((dim >> 5) & 3))); };
    // staging: this thread's K chunks, and 4 positions x 8 dims of V
    const __half *kbase = p.kc + (size_t)kvh * HD, *vbase = p.vc + (size_t)kvh * HD;
    size_t koff[KU];
#pragma unroll
    for (int i = 0; i < KU; i++) {
        const int u = tid + 256 * i, row = u / C;
        koff[i] = (size_t)row * p.kv_dim + 8 * swz(row, u % C);
    }
    const int dc = tid % C, pg = tid / C;
    const bool vthread = pg < 16;
    uint4 vr[4];
    auto stage_k = [&](auto q, uint32_t page) {
        const size_t row0 = (size_t)page << 6;
#pragma unroll
        for (int i = 0; i < KU; i++)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(kbase + row0 * p.kv_dim + koff[i]),
                (__attribute__((address_space(3))) void *)((decltype(q)::value ? ks1 : ks0) + 64 * wave + 256 * i), 16, 0, 0);
    };
    auto load_v = [&](uint32_t page) {
        const size_t row0 = (size_t)page << 6;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = min(4 * pg + i, 63);
            vr[i] = *reinterpret_cast<const uint4 *>(vbase + (row0 + r) * p.kv_dim + 8 * dc);
        }
    };
    auto put = [&](auto q, int t) {
        uint2 *vs = decltype(q)::value ? vs1 : vs0;
        // positions past the pass's last hold no row yet: zeros, so that their weight 0 adds 0
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (64 * t + 4 * pg + i > kv_last) vr[i] = uint4{0, 0, 0, 0};
        const uint32_t a[4][4] = {{vr[0].x, vr[0].y, vr[0].z, vr[0].w}, {vr[1].x, vr[1].y, vr[1].z, vr[1].w},
                                  {vr[2].x, vr[2].y, vr[2].z, vr[2].w}, {vr[3].x, vr[3].y, vr[3].z, vr[3].w}};
        if (vthread)
#pragma unroll
            for (int d = 0; d < 8; d++) {
                const uint32_t sel = (d & 1) ? 0x07060302u : 0x05040100u;
                vs[vslot(8 * dc + d, pg)] = {__builtin_amdgcn_perm(a[1][d >> 1], a[0][d >> 1], sel),
                                             __builtin_amdgcn_perm(a[3][d >> 1], a[2][d >> 1], sel)};
            }
    };

    // the queries as pieces, B operands
    ph8 qh[KT], ql[KT];
    {
        const float *qr = p.q + (size_t)qc * p.q_stride + (size_t)(kvh * p.G + (valid ? v % p.G : 0)) * HD;
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const float4 x = *reinterpret_cast<const float4 *>(qr + 16 * t + 8 * lh),
                         y = *reinterpret_cast<const float4 *>(qr + 16 * t + 8 * lh + 4);
            const float f[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float s = f[e] * p.qscale;
                qh[t][e] = (_Float16)s;
                ql[t][e] = (_Float16)(s - (float)qh[t][e]);
            }
        }
    }
    pf16 o[DT];
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[d][r] = 0.f;
    float m = -INFINITY, l = 0.f;

    // a row that sees none of its split's positions has no maximum yet: its weights are exp2(-inf) = 0
    auto finite = [](float v) { return v == -INFINITY ? 0.f : v; };
    uint32_t page1 = p.pages[min(t_begin + 1, nt - 1)];  // the next tile's page
    auto compute = [&](auto q, int t, bool more) {
        const uint4 *ks = decltype(q)::value ? ks1 : ks0;
        const uint2 *vs = decltype(q)::value ? vs1 : vs0;
        // byte offsets of this lane's reads: a row's start and the exchange's low bits; hidden from
        // the optimiser, which would otherwise keep every exchanged address in a register
        uint32_t kb = l32 * (16 * C) + 16 * (HD == 96 ? lh : swz(l32, lh)), vb = l32 * 128 + 8 * (lh ^ (l32 >> 1));
        asm("" : "+v"(kb), "+v"(vb));
        pf16 s[2];
#pragma unroll
        for (int pt = 0; pt < 2; pt++) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[pt][r] = 0.f;
#pragma unroll
            for (int k = 0; k < KT; k++) {
                const uint32_t at = (HD == 96 ? kb + 32 * k : kb ^ (32 * k)) + pt * (512 * C);
                const ph8 a = *reinterpret_cast<const ph8 *>(reinterpret_cast<const char *>(ks) + at);
                s[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[k], s[pt], 0, 0, 0);
                s[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[k], s[pt], 0, 0, 0);
            }
        }
        // the next tile's V into registers while the softmax and the value products run
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_v(page1);
        __builtin_amdgcn_sched_barrier(0);
        if (64 * t + 63 > wave_first) {
            const int lim = qpos - 64 * t - 4 * lh;
#pragma unroll
            for (int pt = 0; pt < 2; pt++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (32 * pt + 8 * (r >> 2) + (r & 3) > lim) s[pt][r] = -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int r = 1; r < 32; r++) mx = fmaxf(mx, s[r >> 4][r & 15]);
        mx = pair_max(mx);
        if (__any(mx > m)) {
            const float mn = fmaxf(m, mx), al = __builtin_amdgcn_exp2f(m - finite(mn));
            m = mn;
            l *= al;
#pragma unroll
            for (int d = 0; d < DT; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[d][r] *= al;
        }
        const float mf = finite(m);
#pragma unroll
        for (int pt = 0; pt < 2; pt++) {
            uint32_t hi[8], lo[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float a = __builtin_amdgcn_exp2f(s[pt][2 * i] - mf), b = __builtin_amdgcn_exp2f(s[pt][2 * i + 1] - mf);
                l += a + b;
                // (the packed multiply is exact, and half the instructions of scaling a and b)
                const ph2 h = ph2{(_Float16)a, (_Float16)b} * (_Float16)kPaWeight;
                const ph2 w = {(_Float16)fmaf(a, kPaWeight, -(float)h[0]), (_Float16)fmaf(b, kPaWeight, -(float)h[1])};
                hi[i] = __builtin_bit_cast(uint32_t, h);
                lo[i] = __builtin_bit_cast(uint32_t, w);
            }
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const ph8 ph = __builtin_bit_cast(ph8, uint4{hi[4 * k], hi[4 * k + 1], hi[4 * k + 2], hi[4 * k + 3]}),
                          pl = __builtin_bit_cast(ph8, uint4{lo[4 * k], lo[4 * k + 1], lo[4 * k + 2], lo[4 * k + 3]});
#pragma unroll
                for (int d = 0; d < DT; d++) {
                    // granules 8 pt + 4 k + lh and two on, of dim 32 d + l32 (vslot)
                    const char *vd = reinterpret_cast<const char *>(vs) + 4096 * d;
                    const uint2 x = *reinterpret_cast<const uint2 *>(vd + (vb ^ (8 * ((8 * pt + 4 * k) ^ d)))),
                                y = *reinterpret_cast<const uint2 *>(vd + (vb ^ (8 * ((8 * pt + 4 * k + 2) ^ d))));
                    const ph8 a = __builtin_bit_cast(ph8, uint4{x.x, x.y, y.x, y.y});
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph, o[d], 0, 0, 0);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl, o[d], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    if (t_begin >= nt) return;  // (the launch has at most one split per tile of the shortest range)
    stage_k(c0, p.pages[t_begin]);
    load_v(p.pages[t_begin]);
    put(c0, t_begin);
    __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    auto tile = [&](auto q, int t) {
        constexpr std::integral_constant<int, 1 - decltype(q)::value> other{};
        const bool more = t + 1 < nt;
        const uint32_t page2 = p.pages[min(t + 2, nt - 1)];
        if (more) stage_k(other, page1);
        compute(q, t, more);
        if (more) put(other, t + 1);
        page1 = page2;
        __builtin_amdgcn_s_waitcnt(0x70);
        __builtin_amdgcn_s_barrier();
    };
    for (int t = t_begin; t < nt; t += 2) {
        tile(c0, t);
        if (t + 1 < nt) tile(c1, t + 1);
    }
    l = pair_sum(l) * kPaWeight;  // as the outputs
    if (!valid) return;
    const bool split = ks > 1;
    const float inv = split ? 1.f : 1.f / l;
    const int heads = p.G * p.nkv;
    const size_t row = ((size_t)z * p.M + qi) * heads + head;
    float *dst = (split ? p.part + row * HD : p.out + (size_t)qi * p.out_stride + (size_t)head * HD) + 4 * lh;
#pragma unroll
    for (int d = 0; d < DT; d++)
#pragma unroll
        for (int g = 0; g < 4; g++)
            *reinterpret_cast<float4 *>(dst + 32 * d + 8 * g) = make_float4(
                o[d][4 * g] * inv, o[d][4 * g + 1] * inv, o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv);
    if (split && lh == 0) *reinterpret_cast<float2 *>(p.part_ml + row * 2) = make_float2(m, l);
}

// The splits' partial outputs of a (query, head) row, in their order; a thread per four dims.
template <int HD>
__global__ void __launch_bounds__(256) pattn_merge_kernel(const float *__restrict__ part, const float *__restrict__ part_ml,
                                                          float *__restrict__ out, int rows, int heads, int out_stride,
                                                          int ks) {
    const int i = blockIdx.x * 256 + threadIdx.x, row = i / (HD / 4), d = 4 * (i % (HD / 4));
    if (row >= rows) return;
    float m = -INFINITY;
    for (int z = 0; z < ks; z++) m = fmaxf(m, part_ml[((size_t)z * rows + row) * 2]);
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    float l = 0.f;
    for (int z = 0; z < ks; z++) {
        const size_t r = (size_t)z * rows + row;
        const float2 ml = *reinterpret_cast<const float2 *>(part_ml + r * 2);
        const float w = ml.x == -INFINITY && m != -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - m);
        const float4 v = *reinterpret_cast<const float4 *>(part + r * HD + d);
        a.x = fmaf(w, v.x, a.x), a.y = fmaf(w, v.y, a.y), a.z = fmaf(w, v.z, a.z), a.w = fmaf(w, v.w, a.w);
        l = fmaf(w, ml.y, l);
    }
    const float inv = 1.f / l;
    *reinterpret_cast<float4 *>(out + (size_t)(row / heads) * out_stride + (size_t)(row % heads) * HD + d) =
        make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
}

bool prompt_attention_supported(int head_dim, int head_count, int head_count_kv) {
    return (head_dim == 64 || head_dim == 96 || head_dim == 128) && head_count_kv > 0 && head_count % head_count_kv == 0 &&
           head_count / head_count_kv <= kPaRows;
}

hipError_t launch_prompt_attention(const AttnParams &a, float *part, size_t part_floats, hipStream_t s) {
    if (!prompt_attention_supported(a.head_dim, a.head_count, a.head_count_kv) || a.n_query < 1 || a.position_dev ||
        a.position < 0 || a.position + a.n_query > a.ctx || a.window_start != 0 || !a.page_table || a.page_shift != 6 ||
        a.kv_dim % 8 || a.q_stride % 4 || a.out_stride % 4 || ((uintptr_t)a.q | (uintptr_t)a.out | (uintptr_t)part) % 16 ||
        ((uintptr_t)a.k_cache | (uintptr_t)a.v_cache) % 16)
        return hipErrorInvalidValue;
    PAttnParams p{};
    p.q = a.q, p.out = a.out, p.kc = a.k_cache, p.vc = a.v_cache, p.pages = a.page_table;
    p.M = a.n_query, p.pos = a.position, p.G = a.head_count / a.head_count_kv, p.nkv = a.head_count_kv;
    p.kv_dim = a.kv_dim, p.q_stride = a.q_stride, p.out_stride = a.out_stride;
    p.qn = kPaRows / p.G;
    p.qscale = a.scale * 1.44269504088896340736f;
    const int wgs = p.nkv * ((p.M + p.qn - 1) / p.qn);
    const int first_tiles = ((p.pos + (p.M < p.qn ? p.M : p.qn) - 1) >> 6) + 1;  // of the earliest queries
    const size_t rows = (size_t)p.M * a.head_count;
    int ks = 1;
    while (part && ks < 16 && wgs * ks * 2 <= 512 && first_tiles >= 4 * ks * 2 &&
           rows * (ks * 2) * (a.head_dim + 2) <= part_floats)
        ks *= 2;
    p.part = part, p.part_ml = part ? part + (size_t)ks * rows * a.head_dim : nullptr;
    auto go = [&](auto hd) {
        constexpr int HD = decltype(hd)::value;
        hipLaunchKernelGGL(pattn_kernel<HD>, dim3(wgs, ks), dim3(256), 0, s, p);
        if (ks > 1)
            hipLaunchKernelGGL(pattn_merge_kernel<HD>, dim3((unsigned)((rows * (HD / 4) + 255) / 256)), dim3(256), 0, s,
                               p.part, p.part_ml, p.out, (int)rows, a.head_count, p.out_stride, ks);
    };
    switch (a.head_dim) {
    case 64: go(std::integral_constant<int, 64>{}); break;
    case 96: go(std::integral_constant<int, 96>{}); break;
    case 128: go(std::integral_constant<int, 128>{}); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace zh
