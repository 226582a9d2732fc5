// zh_pgemm.hip -- the prompt passes' products: many token rows against a
// quantized matrix on the f16 matrix cores.
//
//   Y[m][n] (=, +=) sum_k W[n][k] X[m][k]        (or silu(gate) * up of two matrices)
//
// Codes.  Within a 256-value block a weight is d_block * c with c = scale * code a small integer
// (Q4_K: at most 945, less dmin * m_j per 32 values; Q3_K: 128; Q8_0: 127, its d per 32 values),
// so c is exact in binary16.  Q6_K's and IQ4_XS's c (up to 4096) take two pieces, c = hi + lo
// exactly.  The activations come as hi + lo pieces of rows scaled by a power of two (HPlanes).
// A product is x_hi c + x_lo c (+ x_hi c_lo): the weights are never rounded and x to 2^-22; two
// (three) matrix products per weight instead of the rounded weight's one.
//
// Units.  The accumulators are in units of the current block's d: at a block's first slab they are
// multiplied by d_before / d_now per column (one multiply per result and 256 values, where adding
// each block's product by an FMA would need a second set of accumulators), for Q4_K by way of dmin,
// in whose units the minimum terms -m_j * (sum of 32 x) are one product of the same kind.  A change
// of unit rounds each result once (twice a block for Q4_K, once every 32 values for Q8_0), as an FMA
// per block would; the factors' own roundings don't add up (unit_to): 14336 Q8_0 values whose scales
// alternate are 8.8e-7 from 64 bits (relative 2-norm; 3.8e-6 with plain quotients), random scales
// 8.2e-7, bf16 pieces and an FMA per block 2.4e-6.  A block with d = 0 adds nothing and leaves the
// unit as it was.
//
// Layout.  A workgroup takes TM tokens x TN rows; a wavefront 32 WM x 32 WN on 32x32x16 products
// (A = activations, B = codes: lane l holds row l % 32's results, so a column's factor is one
// value per lane).  A slab is 32 values: its activations go to LDS by the asynchronous copy, each
// thread decodes 16 codes of a row into LDS, two slabs deep, one barrier per slab.  Chunks of 16
// bytes are exchanged within 256 bytes of rows so that the 16 lanes of a read cover all banks.
// Half of the wavefronts decode before their products and half after, so that the two of a SIMD
// take turns; decoding ahead of the next loads keeps the wait for the codes from waiting for them.
//
// What bounds it: 256 x 256 tiles at 4095 x 4096 x 14336 (Q4_K) take 1075 us, 450 TFLOP/s of the
// product, 900 of issued matrix work, where the library's f16 product reaches 1180-1230 on the same
// card (its clock falls to 1.95 GHz under this load); a slab takes about 4100 cycles of which the
// matrix cores are busy 2048.  The same wait for codes and loads together took 1300 us, without
// the asynchronous copy 1293 us with one slab in registers.
#include <type_traits>

#include "zh_internal.h"
#include "zh_quant.h"

namespace zh {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ h2v as_h2(uint32_t v) { return __builtin_bit_cast(h2v, v); }
__device__ __forceinline__ uint32_t as_u(h2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2v splat(float v) {
    const _Float16 h = (_Float16)v;
    return h2v{h, h};
}
// unsigned bytes 0, 1 (hi 0) or 2, 3 (hi 1) of c as the binary16 pair 1024 + c
template <int HI> __device__ __forceinline__ h2v b1024(uint32_t c) {
    return as_h2(__builtin_amdgcn_perm(0x64646464u, c, HI ? 0x04030402u : 0x04010400u));
}

// ---- per-format staging: 16 consecutive codes of one row per thread ----
// load: the bytes of stage j (0 .. 7: values 32 j .. of block row b), half h (values 16 h ..);
// decode: hi (and lo) pieces of the integer codes; unit: the block's scale.
template <int F> struct PFmt;

template <> struct PFmt<Q4_K> {
    static constexpr int kBytes = 144;
    static constexpr bool kLo = false, kMin = true, kUnit32 = false;
    uint4 hd, q;
    __device__ __forceinline__ void load(const uint8_t *b, int j, int h) {
        hd = ld16(b);
        q = ld16(b + 16 + 32 * (j >> 1) + 16 * h);
    }
    __device__ __forceinline__ float unit() const { return h2f(hd.x); }
    __device__ __forceinline__ float min_unit() const { return h2f(hd.x >> 16); }
    __device__ __forceinline__ uint32_t sbyte(int k) const {
        const uint32_t w = k < 4 ? hd.y : k < 8 ? hd.z : hd.w;
        return (w >> (8 * (k & 3))) & 0xFFu;
    }
    __device__ __forceinline__ void decode(int j, int h, uint32_t (&hi)[8], uint32_t (&lo)[8]) const {
        const uint32_t sc = j < 4 ? sbyte(j) & 63 : (sbyte(j + 4) & 0x0F) | ((sbyte(j - 4) >> 6) << 4);
        const h2v s = splat((float)sc), off = splat(-1024.f * (float)sc);
        const int sh = 4 * (j & 1);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t c = (w[i] >> sh) & 0x0F0F0F0Fu;
            // (1024 + c) sc - 1024 sc, one rounding: c sc exactly (at most 945)
            hi[2 * i] = as_u(__builtin_elementwise_fma(b1024<0>(c), s, off));
            hi[2 * i + 1] = as_u(__builtin_elementwise_fma(b1024<1>(c), s, off));
        }
    }
    // -64 m_j of the block's eight minimums
    __device__ __forceinline__ uint4 mins(bool live) const {
        float m[8];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t mid = (hd.z >> (8 * j)) & 0xFFu, top = (hd.w >> (8 * j)) & 0xFFu;
            m[j] = live ? -64.f * (float)(mid & 63) : 0.f;
            m[4 + j] = live ? -64.f * (float)((top >> 4) | ((mid >> 6) << 4)) : 0.f;
        }
        uint32_t r[4];
#pragma unroll
        for (int i = 0; i < 4; i++) r[i] = as_u(h2v{(_Float16)m[2 * i], (_Float16)m[2 * i + 1]});
        return {r[0], r[1], r[2], r[3]};
    }
};

template <> struct PFmt<Q8_0> {
    static constexpr int kBytes = 272;  // eight 32-value blocks
    static constexpr bool kLo = false, kMin = false, kUnit32 = true;
    uint4 q;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t *b, int j, int h) {
        d = ld2(b + 34 * j);
        q = ld16(b + 34 * j + 2 + 16 * h);
    }
    __device__ __forceinline__ float unit() const { return h2f(d); }
    __device__ __forceinline__ void decode(int, int, uint32_t (&hi)[8], uint32_t (&lo)[8]) const {
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
        const h2v off = splat(-1152.f);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t c = w[i] ^ 0x80808080u;  // 128 + q
            hi[2 * i] = as_u(b1024<0>(c) + off);
            hi[2 * i + 1] = as_u(b1024<1>(c) + off);
        }
    }
};

// hi = binary16(s v), lo = s v - hi: exact for |s v| <= 4096
__device__ __forceinline__ void two_pieces(h2v v, h2v s, uint32_t &hi, uint32_t &lo) {
    const h2v p = v * s;
    hi = as_u(p);
    lo = as_u(__builtin_elementwise_fma(v, s, -p));
}

template <> struct PFmt<Q6_K> {
    static constexpr int kBytes = 210;
    static constexpr bool kLo = true, kMin = false, kUnit32 = false;
    uint4 ql, qh;
    uint32_t d, sc;
    __device__ __forceinline__ void load(const uint8_t *b, int j, int h) {
        ql = ld16(b + 64 * (j >> 2) + 32 * (j & 1) + 16 * h);
        qh = ld16(b + 128 + 32 * (j >> 2) + 16 * h);
        sc = b[192 + 2 * j + h];
        d = ld2(b + 208);
    }
    __device__ __forceinline__ float unit() const { return h2f(d); }
    __device__ __forceinline__ void decode(int j, int, uint32_t (&hi)[8], uint32_t (&lo)[8]) const {
        const int s4 = 2 * (j & 2), s2 = 2 * (j & 3);
        const uint32_t a[4] = {ql.x, ql.y, ql.z, ql.w}, c[4] = {qh.x, qh.y, qh.z, qh.w};
        const h2v s = splat((float)(int8_t)sc), off = splat(-1056.f);  // 1024 + 32
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v = ((a[i] >> s4) & 0x0F0F0F0Fu) | (((c[i] >> s2) & 0x03030303u) << 4);
            two_pieces(b1024<0>(v) + off, s, hi[2 * i], lo[2 * i]);
            two_pieces(b1024<1>(v) + off, s, hi[2 * i + 1], lo[2 * i + 1]);
        }
    }
};

template <> struct PFmt<IQ4_XS> {
    static constexpr int kBytes = 136;
    static constexpr bool kLo = true, kMin = false, kUnit32 = false;
    uint2 hd;
    uint4 q;
    __device__ __forceinline__ void load(const uint8_t *b, int j, int) {
        hd = ld8(b);
        q = ld16(b + 8 + 16 * j);
    }
    __device__ __forceinline__ float unit() const { return h2f(hd.x); }
    __device__ __forceinline__ void decode(int j, int h, uint32_t (&hi)[8], uint32_t (&lo)[8]) const {
        const uint32_t low = (hd.y >> (4 * j)) & 0x0F, high = (hd.x >> (16 + 2 * j)) & 3;
        const h2v s = splat((float)((int)(low | (high << 4)) - 32)), off = splat(-1152.f);
        const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t c = iq4_lookup4((w[i] >> (4 * h)) & 0x0F0F0F0Fu) ^ 0x80808080u;
            two_pieces(b1024<0>(c) + off, s, hi[2 * i], lo[2 * i]);
            two_pieces(b1024<1>(c) + off, s, hi[2 * i + 1], lo[2 * i + 1]);
        }
    }
};

template <> struct PFmt<Q3_K> {
    static constexpr int kBytes = 110;
    static constexpr bool kLo = false, kMin = false, kUnit32 = false;
    uint4 hm, qs;
    uint32_t sl, sh, d;
    __device__ __forceinline__ void load(const uint8_t *b, int j, int h) {
        hm = ld16(b + 16 * h);
        qs = ld16(b + 32 + 32 * (j >> 2) + 16 * h);
        const int si = 2 * j + h;
        sl = b[96 + (si & 7)];
        sh = b[104 + (si & 3)];
        d = ld2(b + 108);
    }
    __device__ __forceinline__ float unit() const { return h2f(d); }
    __device__ __forceinline__ void decode(int j, int h, uint32_t (&hi)[8], uint32_t (&lo)[8]) const {
        const int si = 2 * j + h;
        const uint32_t s6 = ((sl >> (4 * (si >> 3))) & 0xF) | (((sh >> (2 * (si >> 2))) & 3) << 4);
        const h2v s = splat((float)((int)s6 - 32)), off = splat(-1028.f);  // 1024 + 4
        const uint32_t a[4] = {qs.x, qs.y, qs.z, qs.w}, m[4] = {hm.x, hm.y, hm.z, hm.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t c = ((a[i] >> (2 * (j & 3))) & 0x03030303u) | (((m[i] >> j) & 0x01010101u) << 2);
            hi[2 * i] = as_u((b1024<0>(c) + off) * s);
            hi[2 * i + 1] = as_u((b1024<1>(c) + off) * s);
        }
    }
};

struct PGemmParams {
    const uint8_t *w[3], *w2;  // matrices (w2: up, with SWIGLU)
    float *y[3];
    int N[3], ldy[3], t0[3];   // rows, output row stride, first column tile of each matrix
    uint64_t stride;           // bytes per row
    const uint16_t *x, *xs;    // HPlanes
    const float *xscale;
    int M, K, tiles_m, tiles_n;
    // reduction split over gridDim.y workgroups (whole 256-value blocks): their partial results at
    // part + y Msum, Msum the results of all matrices (matrix i's from poff[i], row stride N[i])
    float *part;
    size_t msum, poff[3];
};

// WM x WN tiles of 32 x 32 (tokens x rows) per wavefront, NM x NN wavefronts.
template <int F, int OUT, int WM, int WN, int NM, int NN>
__global__ void __launch_bounds__(64 * NM * NN, 2) pgemm_kernel(PGemmParams p) {
    using P = PFmt<F>;
    constexpr int T = 64 * NM * NN, TM = 32 * WM * NM, TN = 32 * WN * NN;
    static_assert(TN == T / 2, "a thread stages half a row's 32 codes");
    constexpr bool kPair = OUT == OUT_SWIGLU;
    constexpr int TNO = kPair ? TN / 2 : TN;  // output rows per tile
    constexpr int AU = TM * 8 / T;            // 16-byte units of the activations per thread and stage
    static_assert(TM * 8 % T == 0, "whole units per thread");
    constexpr int BROW = P::kLo ? 8 : 4;      // 16-byte chunks of a staged code row
    // two slabs of each, as objects of their own: the wait for the slab on the way is then
    // not taken before the reads of the other
    __shared__ __align__(16) uint4 as0[TM * 8], as1[TM * 8], bs0[TN * BROW], bs1[TN * BROW];
    __shared__ __align__(16) uint4 mas[P::kMin ? TM * 2 : 1], mbs[P::kMin ? TN : 1];
    __shared__ float r1s[P::kMin ? TN : 1], r2s[2][TN];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, lh = lane >> 5;
    const int wm = wave % NM, wn = wave / NM;
    // tile of this workgroup: consecutive tiles of one XCD share rows and tokens
    int mt, nt;
    {
        const int n = p.tiles_m * p.tiles_n, id = blockIdx.x, xcd = id & 7, q = n >> 3, r = n & 7;
        const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (id >> 3);
        constexpr int GM = 4;
        const int per = GM * p.tiles_n, g = t / per, in = t - g * per, gm = min(GM, p.tiles_m - g * GM);
        mt = g * GM + in % gm;
        nt = in / gm;
    }
    const int m0 = mt * TM;
    int seg = 0;
    if (nt >= p.t0[1]) seg = 1;
    if (nt >= p.t0[2]) seg = 2;
    const int N = p.N[seg], n0 = (nt - p.t0[seg]) * TNO;

    // staging: this thread's code row and half
    const int brow = tid >> 1, bh = tid & 1;
    const uint8_t *wrow;
    {
        const uint8_t *w = p.w[seg];
        int row = n0 + brow;
        if (kPair) {
            constexpr int WC = 32 * WN;  // rows of a wavefront column: gate rows, then the same up rows
            const int c = brow / WC, in = brow % WC;
            if (in >= WC / 2) w = p.w2;
            row = n0 + c * (WC / 2) + in % (WC / 2);
        }
        wrow = w + (uint64_t)min(row, N - 1) * p.stride;
    }
    // activations go to LDS without passing registers: unit u of a slab's tile (16 bytes of
    // token row u / 8) takes the chunk that the swizzled image holds there
    const uint16_t *xp[AU];
#pragma unroll
    for (int i = 0; i < AU; i++) {
        const int u = tid + i * T, row = u >> 3, c = (u & 7) ^ ((row >> 1) & 7);
        xp[i] = p.x + (size_t)min(m0 + row, p.M - 1) * 64 + 8 * c;
    }
    const size_t xstep = (size_t)p.M * 64;  // one 32-value slab of every row
    // slabs [s_begin, S): whole 256-value blocks
    const int nblk = p.K >> 8, ks = gridDim.y, z = blockIdx.y;
    const int s_begin = 8 * (int)((long long)z * nblk / ks), S = 8 * (int)((long long)(z + 1) * nblk / ks);

    P raw;
    uint4 msr{};
    auto load_a = [&](auto q, int s) {
#pragma unroll
        for (int i = 0; i < AU; i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(xp[i] + s * xstep),
                                             (__attribute__((address_space(3))) void *)((decltype(q)::value ? as1 : as0) + 64 * wave + i * T), 16, 0, 0);
    };
    auto load_b = [&](int s) {
        raw.load(wrow + (size_t)(s >> 3) * P::kBytes, s & 7, bh);
        if constexpr (P::kMin) {
            // the block's 32-value sums of token row tid / 2
            const int row = min(tid >> 1, TM - 1);
            if ((s & 7) == 0)
                msr = *reinterpret_cast<const uint4 *>(p.xs + ((size_t)(s >> 3) * p.M + min(m0 + row, p.M - 1)) * 16 + 8 * (tid & 1));
        }
    };
    // The accumulators' unit (of row brow; the threads that store its factors).  A factor is a rounded
    // quotient; what it leaves, `carry` of the unit, goes into the next one, so that the product of
    // any run of factors is off by about one rounding and not by one for each.
    float u_prev = 1.f, carry = 0.f;
    auto unit_to = [&](float d) {
        const float r = fmaf(carry, u_prev, u_prev) / d;
        const float left = carry + fmaf(-r, d, u_prev) * __builtin_amdgcn_rcpf(u_prev);
        carry = fabsf(left) < 1e-6f ? left : 0.f;  // (0 where a scale is not finite)
        u_prev = d;
        return r;
    };
    auto store = [&](auto q, int s) {
        constexpr int buf = decltype(q)::value;
        const int j = s & 7;
        const float d = raw.unit();
        const bool live = d != 0.f;
        const uint32_t mask = live ? 0xFFFFFFFFu : 0u;
        uint32_t hi[8], lo[8];
        raw.decode(j, bh, hi, lo);
        uint4 *row = (buf ? bs1 : bs0) + brow * BROW;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const uint4 v = {hi[4 * c] & mask, hi[4 * c + 1] & mask, hi[4 * c + 2] & mask, hi[4 * c + 3] & mask};
            if constexpr (P::kLo) {
                const uint4 v2 = {lo[4 * c] & mask, lo[4 * c + 1] & mask, lo[4 * c + 2] & mask, lo[4 * c + 3] & mask};
                row[(2 * bh + c) ^ ((brow >> 1) & 7)] = v;
                row[(4 + 2 * bh + c) ^ ((brow >> 1) & 7)] = v2;
            } else {
                row[(2 * bh + c) ^ ((brow >> 2) & 3)] = v;
            }
        }
        if (P::kUnit32 || j == 0) {
            if constexpr (P::kMin) {
                const float dm = raw.min_unit();
                const bool ml = dm != 0.f;
                if (bh == 0) {
                    r1s[brow] = ml ? unit_to(dm) : 1.f;
                    mbs[brow] = raw.mins(ml);
                }
                if (tid < 2 * TM) mas[tid] = msr;
            }
            if (bh == 0) r2s[P::kUnit32 ? buf : 0][brow] = live ? unit_to(d) : 1.f;
        }
    };

    f16v acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; i++)
#pragma unroll
        for (int j = 0; j < WN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
    auto scale_cols = [&](const float *rs) {
#pragma unroll
        for (int j = 0; j < WN; j++) {
            const float r = rs[(wn * WN + j) * 32 + l32];
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int q = 0; q < 16; q++) acc[i][j][q] *= r;
        }
    };
    auto compute = [&](auto pq, int s) {
        constexpr int buf = decltype(pq)::value;
        const uint4 *as = buf ? as1 : as0, *bs = buf ? bs1 : bs0;
        if (P::kUnit32 || (s & 7) == 0) {
            if constexpr (P::kMin) {
                scale_cols(r1s);
                h8v ma[WM], mb[WN];
#pragma unroll
                for (int i = 0; i < WM; i++) ma[i] = __builtin_bit_cast(h8v, mas[((wm * WM + i) * 32 + l32) * 2 + lh]);
#pragma unroll
                for (int j = 0; j < WN; j++) mb[j] = __builtin_bit_cast(h8v, mbs[(wn * WN + j) * 32 + l32]);
#pragma unroll
                for (int i = 0; i < WM; i++)
#pragma unroll
                    for (int j = 0; j < WN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ma[i], mb[j], acc[i][j], 0, 0, 0);
            }
            scale_cols(r2s[P::kUnit32 ? buf : 0]);
        }
        h8v a[2][WM][2], b[2][WN], bl[2][P::kLo ? WN : 1];
        auto frags = [&](int t) {
#pragma unroll
            for (int i = 0; i < WM; i++) {
                const int row = (wm * WM + i) * 32 + l32;
#pragma unroll
                for (int q = 0; q < 2; q++)
                    a[t][i][q] = __builtin_bit_cast(h8v, as[row * 8 + ((4 * q + 2 * t + lh) ^ ((row >> 1) & 7))]);
            }
#pragma unroll
            for (int j = 0; j < WN; j++) {
                const int row = (wn * WN + j) * 32 + l32;
                if constexpr (P::kLo) {
                    b[t][j] = __builtin_bit_cast(h8v, bs[row * 8 + ((2 * t + lh) ^ ((row >> 1) & 7))]);
                    bl[t][j] = __builtin_bit_cast(h8v, bs[row * 8 + ((4 + 2 * t + lh) ^ ((row >> 1) & 7))]);
                } else {
                    b[t][j] = __builtin_bit_cast(h8v, bs[row * 4 + ((2 * t + lh) ^ ((row >> 2) & 3))]);
                }
            }
        };
        auto mults = [&](int t) {
#pragma unroll
            for (int q = 0; q < 2; q++)
#pragma unroll
                for (int i = 0; i < WM; i++)
#pragma unroll
                    for (int j = 0; j < WN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][i][q], b[t][j], acc[i][j], 0, 0, 0);
            if constexpr (P::kLo) {
#pragma unroll
                for (int i = 0; i < WM; i++)
#pragma unroll
                    for (int j = 0; j < WN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t][i][0], bl[t][j], acc[i][j], 0, 0, 0);
            }
        };
        frags(0);
        mults(0);
        frags(1);
        mults(1);
    };

    load_b(s_begin);
    load_a(std::integral_constant<int, 0>{}, s_begin);
    store(std::integral_constant<int, 0>{}, s_begin);
    load_b(s_begin + 1);
    __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    // half of the wavefronts stage the next slab before they compute, the
    // others after: the two of a SIMD take turns on its matrix core
    const bool first = wave < NM * NN / 2;
    // slab s is staged in buffer s & 1; raw holds slab s + 1's codes
    auto slab = [&](auto q, int s) {
        constexpr std::integral_constant<int, 1 - decltype(q)::value> o{};
        const bool more = s + 1 < S;
        if (first && more) {
            store(o, s + 1);
            load_b(min(s + 2, S - 1));
        }
        if (more) load_a(o, s + 1);
        compute(q, s);
        __builtin_amdgcn_sched_barrier(0);
        if (!first && more) {
            store(o, s + 1);
            // the copies have landed before the next codes are asked for, which may then stay on their
            // way over the barrier
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            __builtin_amdgcn_sched_barrier(0);
            load_b(min(s + 2, S - 1));
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        } else {
            __builtin_amdgcn_s_waitcnt(0x70);
        }
        __builtin_amdgcn_s_barrier();
    };
    for (int s = s_begin; s < S; s += 2) {
        slab(std::integral_constant<int, 0>{}, s);
        slab(std::integral_constant<int, 1>{}, s + 1);
    }
    __syncthreads();
    // the rows' last units, then y = acc * unit * token scale
    if (bh == 0) r2s[0][brow] = fmaf(carry, u_prev, u_prev);
    __syncthreads();
    scale_cols(r2s[0]);
    // all loads of a group of rows before its stores, none under a branch
    const int nb = kPair ? n0 + wn * (16 * WN) + l32 : n0 + wn * WN * 32 + l32;
    constexpr int NJ = kPair ? WN / 2 : WN;
    const bool split = p.part != nullptr;
    float *const y = split ? p.part + z * p.msum + p.poff[seg] : p.y[seg];
    const int ldy = split ? N : p.ldy[seg];
    const size_t up_off = (size_t)p.M * N;  // the up results follow the gate results in a partial
#pragma unroll
    for (int i = 0; i < WM; i++) {
        const int mb = m0 + (wm * WM + i) * 32 + 4 * lh;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float sc[4], old[4][NJ];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = min(mb + 8 * q + r, p.M - 1);
                sc[r] = p.xscale[m];
                if (OUT == OUT_ADD)
#pragma unroll
                    for (int j = 0; j < NJ; j++) old[r][j] = y[(size_t)m * ldy + min(nb + 32 * j, N - 1)];
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mb + 8 * q + r;
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    const int n = nb + 32 * j;
                    float v = acc[i][j][4 * q + r] * sc[r];
                    if constexpr (kPair) {
                        const float u = acc[i][j + WN / 2][4 * q + r] * sc[r];
                        if (split) {
                            if (m < p.M && n < N) y[up_off + (size_t)m * ldy + n] = u;
                        } else {
                            v = (v / (1.0f + expf(-v))) * u;
                        }
                    }
                    if (OUT == OUT_ADD && !split) v = old[r][j] + v;
                    if (m < p.M && n < N) y[(size_t)m * ldy + n] = v;
                }
            }
        }
    }
}

// The split reduction's partial results, added in their order: y (=, +=) the sum, or
// silu(gate sum) * up sum; one thread per result.
template <int OUT>
__global__ void __launch_bounds__(256) pgemm_reduce_kernel(const float *__restrict__ part, size_t msum, int ks, float *y,
                                                           int ldy, int M, int N) {
    const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (n >= N) return;
    const float *src = part + (size_t)m * N + n;
    float v = 0.f, u = 0.f;
    for (int z = 0; z < ks; z++) {
        v += src[z * msum];
        if (OUT == OUT_SWIGLU) u += src[z * msum + (size_t)M * N];
    }
    float *dst = y + (size_t)m * ldy + n;
    if (OUT == OUT_SWIGLU) v = (v / (1.0f + expf(-v))) * u;
    if (OUT == OUT_ADD) v = *dst + v;
    *dst = v;
}

typedef void (*PGemmKernel)(PGemmParams);
// Tiles.  256 x 256 has the least LDS and L2 traffic per product but one workgroup per CU; 128 x
// 128 and 64 x 128 fill the chip for fewer rows.  Where the tiles still leave CUs idle the
// reduction is split over up to 16 workgroups (partial results added by a second launch in a
// fixed order).  The choice is the least estimate of time: rounds of workgroups over the chip x
// slabs x the measured time of a slab (us; alone on a CU, and with the CU shared or the whole chip
// busy), 6 us for the launch, and the partial results' traffic.  The slab times are Q4_K's; a format
// with a third product per code (Q6_K, IQ4_XS) scales them alike.  Measured against every tile and
// split, 76 / 256 / 600 / 1200 / 4095 rows: 4096 x 4096 Q4_K 29 / 41 / 82 / 128 / 260 us, within 3% of
// the best, Q6_K 33 / 50 / 108 / 188 / 369 and IQ4_XS 31 / 48 / 105 / 173 / 353 within 5%, Q8_0 7%, Q3_K
// 12% (256 rows).  1024 x 4096: within 11% up to 256 rows, 7-19% at 600 and 1200; at 4095 rows 64 x 128
// unsplit is taken where 256 x 256 in four parts would be 1.14-1.33 times as fast (the estimate
// charges the partial results too much there).
struct PTile {
    int tm, tn, threads, per_cu;  // tile, workgroup size, workgroups that share a CU
};
constexpr PTile kPTiles[] = {{256, 256, 512, 1}, {128, 128, 256, 2}, {64, 128, 256, 2}};
template <int F, int OUT> static PGemmKernel pick_pg(int cfg) {
    switch (cfg) {
    case 0: return pgemm_kernel<F, OUT, 2, 4, 4, 2>;
    case 1: return pgemm_kernel<F, OUT, 2, 2, 2, 2>;
    case 2: return pgemm_kernel<F, OUT, 1, 2, 2, 2>;
    default: return nullptr;
    }
}
template <int OUT> static PGemmKernel pick_pgf(int fmt, int cfg) {
    switch (fmt) {
    case Q4_K: return pick_pg<Q4_K, OUT>(cfg);
    case Q6_K: return pick_pg<Q6_K, OUT>(cfg);
    case Q8_0: return pick_pg<Q8_0, OUT>(cfg);
    case IQ4_XS: return pick_pg<IQ4_XS, OUT>(cfg);
    case Q3_K: return pick_pg<Q3_K, OUT>(cfg);
    default: return nullptr;
    }
}

struct PgPlan {
    int cfg, ks;  // tile (kPTiles), reduction split
};
static PgPlan pgemm_plan(int nseg, const int *N, int M, int K, int mats, size_t part_floats) {
    size_t msum = 0;  // partial results of one split
    for (int i = 0; i < nseg; i++) msum += (size_t)mats * M * N[i];
    int cfg = 0, ks = 1;
    double best = 0.0;
    for (int c = 0; c < 3; c++) {
        const PTile &t = kPTiles[c];
        const int tno = t.tn / mats;
        long long tiles = 0;
        for (int i = 0; i < nseg; i++) tiles += (N[i] + tno - 1) / tno;
        tiles *= (M + t.tm - 1) / t.tm;
        for (int k = 1; k <= 16 && k <= K / 256; k *= 2) {
            if (k > 1 && msum * k > part_floats) break;
            static const double one[] = {1.68, 0.85, 0.6}, full[] = {2.43, 1.49, 0.8};
            const long long wgs = tiles * k, slots = 256 * t.per_cu, rounds = (wgs + slots - 1) / slots;
            const double stages = 8.0 * ((K / 256 + k - 1) / k);
            const double cost = rounds * (stages * (wgs <= 256 ? one[c] : full[c]) + 6.0) +
                                (k > 1 ? 4.0 + (double)msum * 4.0 * (2 * k + 1) / 3.0e6 : 0.0);
            if (best == 0.0 || cost < best) best = cost, cfg = c, ks = k;
        }
    }
    return {cfg, ks};
}

bool pgemm_supported(int fmt, int K, const void *w, uint64_t stride) {
    return qgemm_enabled() && qgemm_supported(fmt, K, w, nullptr, stride, 0);
}

hipError_t launch_pgemm(int fmt, int nseg, const uint8_t *const *w, const uint8_t *w2, float *const *y, const int *ldy,
                        const int *N, uint64_t stride, const HPlanes &xp, int M, int K, int out, float *part,
                        size_t part_floats, hipStream_t s) {
    if (nseg < 1 || nseg > 3 || M < 1 || !xp.x || !xp.xs || !xp.scale || (out == OUT_SWIGLU && (nseg != 1 || !w2)) ||
        (out != OUT_STORE && out != OUT_ADD && out != OUT_SWIGLU))
        return hipErrorInvalidValue;
    for (int i = 0; i < nseg; i++)
        if (N[i] < 1 || ldy[i] < N[i] || !y[i] || !pgemm_supported(fmt, K, w[i], stride)) return hipErrorInvalidValue;
    if (w2 && !pgemm_supported(fmt, K, w2, stride)) return hipErrorInvalidValue;
    const int mats = out == OUT_SWIGLU ? 2 : 1;
    PGemmParams p{};
    for (int i = 0; i < nseg; i++) {
        p.w[i] = w[i], p.y[i] = y[i], p.N[i] = N[i], p.ldy[i] = ldy[i];
        p.poff[i] = p.msum;
        p.msum += (size_t)mats * M * N[i];
    }
    p.w2 = w2;
    p.stride = stride;
    p.x = xp.x, p.xs = xp.xs, p.xscale = xp.scale;
    p.M = M, p.K = K;
    const auto [cfg, ks] = pgemm_plan(nseg, N, M, K, mats, part ? part_floats : 0);
    const PTile &t = kPTiles[cfg];
    int nt = 0;
    for (int i = 0; i < 3; i++) {
        p.t0[i] = i < nseg ? nt : 0x7fffffff;
        if (i < nseg) nt += (N[i] + t.tn / mats - 1) / (t.tn / mats);
    }
    p.tiles_m = (M + t.tm - 1) / t.tm, p.tiles_n = nt;
    p.part = ks > 1 ? part : nullptr;
    PGemmKernel k = out == OUT_STORE ? pick_pgf<OUT_STORE>(fmt, cfg)
                    : out == OUT_ADD ? pick_pgf<OUT_ADD>(fmt, cfg)
                                     : pick_pgf<OUT_SWIGLU>(fmt, cfg);
    if (!k) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3(p.tiles_m * p.tiles_n, ks), dim3(t.threads), 0, s, p);
    for (int i = 0; i < nseg && ks > 1; i++) {
        auto red = out == OUT_STORE ? pgemm_reduce_kernel<OUT_STORE>
                   : out == OUT_ADD ? pgemm_reduce_kernel<OUT_ADD>
                                    : pgemm_reduce_kernel<OUT_SWIGLU>;
        hipLaunchKernelGGL(red, dim3((N[i] + 255) / 256, M), dim3(256), 0, s, part + p.poff[i], p.msum, ks, y[i], ldy[i],
                           M, N[i]);
    }
    return hipGetLastError();
}

// ---- the input planes ----

// The power of two that brings a row's largest magnitude to [2^14, 2^15), and its inverse (rows of
// zeros, or with an infinity: 1).
__device__ __forceinline__ void row_scale(float mx, float &s, float &inv) {
    const int e = (int)(__float_as_uint(mx) >> 23) & 0xFF, c = max(e, 15);
    const bool one = mx == 0.f || e == 255;
    s = one ? 1.f : __uint_as_float((uint32_t)(268 - c) << 23);
    inv = one ? 1.f : __uint_as_float((uint32_t)(c - 14) << 23);
}
// Values 4 i .. 4 i + 3 of row m as scaled pieces; the eight lanes of a 32-value block share its sum.
__device__ __forceinline__ void put_planes(const HPlanes &xp, int M, int m, int i, const float4 &v, float s) {
    const float a[4] = {v.x * s, v.y * s, v.z * s, v.w * s};
    _Float16 h[4], l[4];
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        h[c] = (_Float16)a[c];
        l[c] = (_Float16)(a[c] - (float)h[c]);
        sum += (float)h[c] + (float)l[c];
    }
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    sum += __shfl_xor(sum, 4, 64);
    const int kb = i >> 3, at = 4 * (i & 7);
    uint16_t *d = xp.x + ((size_t)kb * M + m) * 64 + at;
    *reinterpret_cast<uint2 *>(d) = {as_u(h2v{h[0], h[1]}), as_u(h2v{h[2], h[3]})};
    *reinterpret_cast<uint2 *>(d + 32) = {as_u(h2v{l[0], l[1]}), as_u(h2v{l[2], l[3]})};
    if ((i & 7) == 0) {
        sum *= 1.f / 64.f;
        const _Float16 sh = (_Float16)sum, sl = (_Float16)(sum - (float)sh);
        uint16_t *e = xp.xs + ((size_t)(kb >> 3) * M + m) * 16 + (kb & 7);
        e[0] = __builtin_bit_cast(uint16_t, sh);
        e[8] = __builtin_bit_cast(uint16_t, sl);
    }
}
__device__ __forceinline__ float max4(float m, const float4 &v) {
    return fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
}

// One workgroup per row, the row in registers up to 4 J 256 values and read again past them.
// NORM: the row's RMSNorm (rmsNorm, model/loader.zig:3404-3426; also stored to out where set).
template <bool NORM>
__global__ void __launch_bounds__(256) row_planes_kernel(const float *__restrict__ x, int ldx, const float *__restrict__ w,
                                                         float *__restrict__ out, int n, float eps, HPlanes xp) {
    const int tid = threadIdx.x, m = blockIdx.x, M = gridDim.x, n4 = n / 4;
    const float4 *x4 = reinterpret_cast<const float4 *>(x + (size_t)m * ldx), *w4 = reinterpret_cast<const float4 *>(w);
    __shared__ float red[2][4];
    constexpr int J = 8;
    float4 v[J], wv[NORM ? J : 1];
#pragma unroll
    for (int j = 0; j < J; j++) v[j] = x4[min(tid + 256 * j, n4 - 1)];
    if (NORM)
#pragma unroll
        for (int j = 0; j < J; j++) wv[j] = w4[min(tid + 256 * j, n4 - 1)];
    float scale = 1.f;
    if (NORM) {
        float ss = 0.f;
        auto sq = [&](const float4 &a) { ss = fmaf(a.w, a.w, fmaf(a.z, a.z, fmaf(a.y, a.y, fmaf(a.x, a.x, ss)))); };
#pragma unroll
        for (int j = 0; j < J; j++)
            if (tid + 256 * j < n4) sq(v[j]);
        for (int i = tid + 256 * J; i < n4; i += 256) sq(x4[i]);
        for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
        if ((tid & 63) == 0) red[0][tid >> 6] = ss;
        __syncthreads();
        const float tot = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        scale = 1.0f / sqrtf(tot / (float)n + eps);
    }
    auto value = [&](const float4 &a, const float4 &b) {
        return NORM ? make_float4((scale * a.x) * b.x, (scale * a.y) * b.y, (scale * a.z) * b.z, (scale * a.w) * b.w) : a;
    };
    auto far = [&](int i) { return value(x4[i], NORM ? w4[i] : make_float4(0.f, 0.f, 0.f, 0.f)); };
    float mx = 0.f;
#pragma unroll
    for (int j = 0; j < J; j++) {
        v[j] = value(v[j], wv[NORM ? j : 0]);
        if (tid + 256 * j < n4) mx = max4(mx, v[j]);
    }
    for (int i = tid + 256 * J; i < n4; i += 256) mx = max4(mx, far(i));
    for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((tid & 63) == 0) red[1][tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    float s, inv;
    row_scale(mx, s, inv);
    if (tid == 0) xp.scale[m] = inv;
    float4 *o4 = reinterpret_cast<float4 *>(out + (size_t)m * n);
#pragma unroll
    for (int j = 0; j < J; j++)
        if (tid + 256 * j < n4) {  // n is a multiple of 256: whole wavefronts
            put_planes(xp, M, m, tid + 256 * j, v[j], s);
            if (NORM && out) o4[tid + 256 * j] = v[j];
        }
    for (int i = tid + 256 * J; i < n4; i += 256) {
        const float4 a = far(i);
        put_planes(xp, M, m, i, a, s);
        if (NORM && out) o4[i] = a;
    }
}

static bool planes_args_ok(const float *x, int ldx, int rows, int n, const HPlanes &xp) {
    return x && rows > 0 && n > 0 && n % 256 == 0 && ldx % 4 == 0 && ldx >= n && (uintptr_t)x % 16 == 0 && xp.x && xp.xs &&
           xp.scale;
}
hipError_t launch_row_planes(const float *x, int ldx, int rows, int n, const HPlanes &xp, hipStream_t s) {
    if (!planes_args_ok(x, ldx, rows, n, xp)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(row_planes_kernel<false>, dim3(rows), dim3(256), 0, s, x, ldx, nullptr, nullptr, n, 0.f, xp);
    return hipGetLastError();
}
hipError_t launch_norm_planes(const float *x, const float *w, float *out, int rows, int n, float eps, const HPlanes &xp,
                              hipStream_t s) {
    if (!planes_args_ok(x, n, rows, n, xp) || !w || (uintptr_t)w % 16 || (uintptr_t)out % 16) return hipErrorInvalidValue;
    hipLaunchKernelGGL(row_planes_kernel<true>, dim3(rows), dim3(256), 0, s, x, n, w, out, n, eps, xp);
    return hipGetLastError();
}

}  // namespace zh

extern "C" int ziggy_hip_probe_prompt_tiles(const uint32_t *rows, uint32_t count, uint32_t tokens, uint32_t cols, int pair,
                                            size_t workspace_floats, ZiggyHipPromptTiles *out, char *err, size_t err_len) {
    bool ok = rows && out && count >= 1 && count <= 3 && (!pair || count == 1) && tokens >= 1 && tokens <= 1u << 20 &&
              cols >= 256 && cols % 256 == 0 && cols <= 1u << 20;
    int n[3] = {};
    for (uint32_t i = 0; ok && i < count; i++) {
        ok = rows[i] >= 1 && rows[i] <= 1u << 20;
        n[i] = (int)rows[i];
    }
    if (!ok) {
        zh::set_err(err, err_len, "invalid probe_prompt_tiles arguments");
        return ZIGGY_HIP_INVALID_ARGUMENT;
    }
    const zh::PgPlan plan = zh::pgemm_plan((int)count, n, (int)tokens, (int)cols, pair ? 2 : 1, workspace_floats);
    const zh::PTile &t = zh::kPTiles[plan.cfg];
    *out = {(uint32_t)t.tm, (uint32_t)t.tn, (uint32_t)plan.ks};
    return ZIGGY_HIP_OK;
}
