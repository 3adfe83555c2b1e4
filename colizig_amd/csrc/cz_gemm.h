// cz_gemm.h - E4M3 weights times f32 rows on the bf16 matrix cores with every
// bit of the rows: many-token projections (matmulFp8, fp8.zig:215-257) and the
// grouped expert products of prompts past the FP8 form's slots.
//
// An f32 is the sum of three bf16 numbers, each the upper half of what is left
// (8 significant bits at f32's exponent range), and E4M3 is exact in bf16.  So
// every product is exact, a K block (128 columns, one weight scale block) is
// summed in f32 alone and added as tot = fma(blk, s, tot): the f32 kernels'
// products and sums, in another order.  The
// rows are scaled by 2^16 and the weights by 2^-16 on the way, because a bf16
// subnormal ends at 2^-133 where an f32 ends at 2^-149.  Row blocks with an
// element of 2^100 or more are scaled by 1/2 instead (no block sum overflows)
// and flagged: of those, bits below 2^-132 are lost.
//
// The split is done as the rows are staged in LDS, or, where a single wave reads
// a staged row, as it reads it: no pass before the product and no scratch.
//
// Bound: one K block of a 32 x 256 tile is 1,536 cycles of MFMA a SIMD.  In the
// gate/up products of 2000 tokens (two workgroups a CU) the counters give 45% of
// the time in MFMA, each of a SIMD's two waves 23% in vector work (E4M3 to bf16,
// the split, the sums) and 20% waiting for memory or a barrier, and the LDS 30%
// busy: vector work and MFMA hardly overlap.  Two f16 terms (hi + lo, 23 bits, and
// fewer beside elements 2^16 times larger) took 555 us where the layer takes 630;
// the error against 64 bits is 2.2e-7 for 2.4e-7, and of the projections at 385
// tokens 0.9e-7 for 1.3e-7 (the GEMV's: 1.6e-7).  Measured and not kept: loads two
// K blocks ahead, and the weights widened one step ahead or without scheduling
// fences (the same time or up to 4% more).
#pragma once

#include "cz_grouped.h"

typedef __bf16 cz_bf8 __attribute__((ext_vector_type(8)));

#define CZ_GF_UP 0x1p16f     // scale of the rows, undone by the weights'
#define CZ_GF_BIG 0x1p100f   // from here on a row block is scaled by
#define CZ_GF_DOWN 0x1p-1f   // this, and its sums by
#define CZ_GF_F 0x1p17f      // this

// 8 E4M3 bytes -> 8 bf16, times 2^-16, exact (0x7F: NaN).
__device__ __forceinline__ cz_bf8 cz_fp8x8_to_bf16(uint32_t w0, uint32_t w1) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    constexpr float sc = 1.0f / CZ_GF_UP;
    const bf2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w0, sc, false);
    const bf2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w0, sc, true);
    const bf2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w1, sc, false);
    const bf2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)w1, sc, true);
    cz_bf8 r;
    r[0] = p0[0]; r[1] = p0[1]; r[2] = p1[0]; r[3] = p1[1];
    r[4] = p2[0]; r[5] = p2[1]; r[6] = p3[0]; r[7] = p3[1];
    return r;
}

// v = hi + mid + lo, each as words of two bf16.  inf (wave-uniform): there may be
// infinities, which have no lower parts (inf - inf); a NaN stays one in some part.
template <int N>
__device__ __forceinline__ void cz_bf16_split(const float (&v)[N], bool inf, uint32_t (&hi)[N / 2],
                                              uint32_t (&mid)[N / 2], uint32_t (&lo)[N / 2]) {
    float r[N];
    auto take = [&](uint32_t(&out)[N / 2]) {  // the upper halves
#pragma unroll
        for (int i = 0; i < N / 2; ++i)
            out[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, r[2 * i + 1]),
                                           __builtin_bit_cast(uint32_t, r[2 * i]), 0x07060302u);
    };
    auto rest = [&] {  // what they leave, exactly
#pragma unroll
        for (int i = 0; i < N; ++i)
            r[i] = r[i] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r[i]) & 0xffff0000u);
    };
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = v[i];
    take(hi);
    rest();
    if (inf)
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (__builtin_isinf(v[i])) r[i] = 0.0f;
    take(mid);
    rest();
    take(lo);
}

// One wave's part of a tile: MR rows x 64 weight rows, as 32 x 32 x 16 products
// (MR = 32: two subtiles) or 16 x 16 x 32 ones (MR = 16: four).  Lane l holds
// column l % MR of subtile m, rows row(l, i).  The K order inside a block is a
// free permutation: lane group l / MR covers offsets (128 / G) (l / MR) + 8 s at
// step s of NS.
template <int MR>
struct GFWave {
    static constexpr int NSUB = 64 / MR, NV = MR == 32 ? 16 : 4, NS = MR == 32 ? 8 : 4, G = 64 / MR;
    typedef float V __attribute__((ext_vector_type(NV)));
    __device__ static __forceinline__ uint32_t row(uint32_t lane, int i) {
        return MR == 32 ? (i / 4) * 8u + (lane >> 5) * 4u + (i % 4) : (lane >> 4) * 4u + i;
    }
    __device__ static __forceinline__ V mfma(cz_bf8 a, cz_bf8 b, V c) {
        if constexpr (MR == 32)
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};

// One workgroup's tile: its WN x KS waves take the same MR rows and 64 weight
// rows each; KS wave groups take every KS-th K block and their sums are added
// at the end.  RAW (one wave reads a staged row): the rows are staged as f32
// and split where they are read, which keeps two workgroups on a CU; else each
// is split once for the waves that share it.
template <int MR, int WN, int KS>
struct GFLds {
    static constexpr bool RAW = WN == 1;
    static constexpr int RB = MR * KS;                  // K blocks of rows staged per pass
    static constexpr int ALD = RAW ? 512 + 16 : 256 + 16;  // LDS bytes of each (+ 16: rows in distinct bank groups)
    static constexpr int PLANES = RAW ? 1 : 3;
    uint8_t a[PLANES][RB * ALD];
    uint8_t w[WN * KS][64 * CZ_GG_WLD];
    float f[RB];               // undoes the scaling of a flagged pass's row blocks
    uint32_t big[WN * KS];     // staging wave saw an element of CZ_GF_BIG or more
    uint64_t src[MR];          // element offset of each tile row's A row
    uint32_t dst[MR];          // C row, ~0u: padding
};

// tot = the wave's products: weight rows 0-31 are wb[0]'s, 32-63 wb[1]'s (each
// clamped at rmax, scales sr); valid in the kh = 0 waves.
template <int MR, int WN, int KS>
__device__ __forceinline__ void cz_gf_tile(GFLds<MR, WN, KS> &sh, const float *__restrict__ a, uint32_t Kd,
                                           const uint8_t *const (&wb)[2], const uint32_t (&rmax)[2],
                                           const float *const (&sr)[2],
                                           typename GFWave<MR>::V (&tot)[GFWave<MR>::NSUB]) {
    typedef GFWave<MR> W;
    typedef GFLds<MR, WN, KS> L;
    typedef typename W::V V;
    constexpr int NT = 64 * WN * KS, RB = MR * KS;
    constexpr int NA = RB * 16 / NT;  // row blocks per thread (16 lanes each, two float4 a lane)
    constexpr int NW = 8;             // 16-byte weight loads per lane
    static_assert(NA * NT == RB * 16, "tile shape");
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t wn = wave % WN, kh = wave / WN;
    const uint32_t nkb = Kd / 128, nit = (nkb + KS - 1) / KS;
    const uint32_t q = tid & 15;
    // A: thread's row block p is rb = tid / 16 + p NT / 16: row rb % MR of K
    // group rb / MR
    const float *ap[NA];
    uint32_t akh[NA];
#pragma unroll
    for (int p = 0; p < NA; ++p) {
        const uint32_t rb = (tid >> 4) + p * (NT / 16);
        ap[p] = a + sh.src[rb % MR] + 4 * q;
        akh[p] = rb / MR;
    }
    // W: load p is weight rows 8 p + l / 8 of the wave's 64, 16-byte chunk l % 8
    const uint8_t *wp[NW];
#pragma unroll
    for (int p = 0; p < NW; ++p)
        wp[p] = wb[p / 4] + (uint64_t)min(8u * (p % 4) + (lane >> 3), rmax[p / 4]) * Kd + (lane & 7u) * 16u;
    uint8_t *lw = sh.w[kh * WN + wn];
    uint8_t *wst = lw + (lane >> 3) * CZ_GG_WLD + (lane & 7u) * 16u;
    float4 av[NA][2];
    u32x4 wv[NW];
    auto load = [&](uint32_t it) {  // K blocks past the end re-read the last one (never added)
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            const float *s = ap[p] + (uint64_t)min(it * KS + akh[p], nkb - 1) * 128;
            av[p][0] = *(const float4 *)s;
            av[p][1] = *(const float4 *)(s + 64);
        }
        const uint32_t kb = min(it * KS + kh, nkb - 1);
#pragma unroll
        for (int p = 0; p < NW; ++p) wv[p] = *(const u32x4 *)(wp[p] + (uint64_t)kb * 128);
    };
    auto store = [&] {
#pragma unroll
        for (int p = 0; p < NW; ++p) *(u32x4 *)(wst + p * 8 * CZ_GG_WLD) = wv[p];
        float all = 0.0f, up[NA];
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            up[p] = CZ_GF_UP;
#pragma unroll
            for (int i = 0; i < 8; ++i) all = fmaxf(all, __builtin_fabsf(((const float *)av[p])[i]));
        }
        const bool big = __builtin_amdgcn_ballot_w64(all >= CZ_GF_BIG) != 0;  // infinities too
        if (big) {
#pragma unroll
            for (int p = 0; p < NA; ++p) {
                float mx = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) mx = fmaxf(mx, __builtin_fabsf(((const float *)av[p])[i]));
                mx = fmaxf(mx, cz_dpp<0xB1>(mx));
                mx = fmaxf(mx, cz_dpp<0x4E>(mx));
                mx = fmaxf(mx, cz_dpp<0x141>(mx));
                mx = fmaxf(mx, cz_dpp<0x140>(mx));
                if (mx >= CZ_GF_BIG) up[p] = CZ_GF_DOWN;
            }
        }
        if (lane == 0) sh.big[wave] = big;
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            const uint32_t rb = (tid >> 4) + p * (NT / 16);
            if (q == 0) sh.f[rb] = up[p] == CZ_GF_UP ? 1.0f : CZ_GF_F;
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = ((const float *)av[p])[i] * up[p];
            if constexpr (L::RAW) {
                uint8_t *o = sh.a[0] + rb * L::ALD + 16 * q;
                *(float4 *)o = make_float4(v[0], v[1], v[2], v[3]);
                *(float4 *)(o + 256) = make_float4(v[4], v[5], v[6], v[7]);
            } else {
                uint32_t t[3][4];
                cz_bf16_split(v, big, t[0], t[1], t[2]);
#pragma unroll
                for (int k = 0; k < L::PLANES; ++k) {
                    uint8_t *o = sh.a[k] + rb * L::ALD + 8 * q;
                    *(uint2 *)o = make_uint2(t[k][0], t[k][1]);
                    *(uint2 *)(o + 128) = make_uint2(t[k][2], t[k][3]);
                }
            }
        }
    };
    const uint32_t rl = lane & (MR - 1), kg = lane / MR;
    const uint32_t ao = (kh * MR + rl) * L::ALD + kg * ((L::RAW ? 512 : 256) / W::G);  // + 8 s elements
    const uint8_t *lr = lw + rl * CZ_GG_WLD + kg * (128 / W::G);                       // + 8 s: the same K order
    static_assert(WN * KS == 4, "the staging waves' flags are one 16-byte word");
    auto multiply = [&](uint32_t it) {
        const uint32_t kb = it * KS + kh;
        if (KS > 1 && kb >= nkb) return;  // wave-uniform
        const float sc[2] = {cz_const_f32(sr[0] + kb), cz_const_f32(sr[1] + kb)};
        const uint4 bg = *(const uint4 *)sh.big;
        const bool big = __builtin_amdgcn_readfirstlane((int)(bg.x | bg.y | bg.z | bg.w)) != 0;
        V blk[W::NSUB] = {}, low[W::NSUB] = {};
        u32x4 wq[2][W::NSUB];
        cz_bf8 xt[2][3];
        auto fetch_w = [&](int s2) {
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) wq[s2 & 1][m] = *(const u32x4 *)(lr + m * MR * CZ_GG_WLD + 16 * s2);
        };
        auto fetch_a = [&](int s) {
            if constexpr (L::RAW) {
                float v[8];
                *(float4 *)&v[0] = *(const float4 *)(sh.a[0] + ao + 32 * s);
                *(float4 *)&v[4] = *(const float4 *)(sh.a[0] + ao + 32 * s + 16);
                uint32_t t[3][4];
                cz_bf16_split(v, big, t[0], t[1], t[2]);
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    xt[s & 1][k] = __builtin_bit_cast(cz_bf8, u32x4{t[k][0], t[k][1], t[k][2], t[k][3]});
            } else {
#pragma unroll
                for (int k = 0; k < L::PLANES; ++k) xt[s & 1][k] = *(const cz_bf8 *)(sh.a[k] + ao + 16 * s);
            }
        };
        fetch_w(0);
        fetch_a(0);
        fetch_w(1);
#pragma unroll
        for (int s = 0; s < W::NS; ++s) {  // step s + 1's operands are read while step s multiplies
            if (s + 1 < W::NS) fetch_a(s + 1);
            if (s >= 2 && s % 2 == 0 && s / 2 + 1 < W::NS / 2) fetch_w(s / 2 + 1);
            cz_bf8 b[W::NSUB];
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) {
                const u32x4 w = wq[(s >> 1) & 1][m];
                b[m] = (s & 1) ? cz_fp8x8_to_bf16(w[2], w[3]) : cz_fp8x8_to_bf16(w[0], w[1]);
            }
            // the lower parts' sum is rounded into the rest once
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) low[m] = W::mfma(xt[s & 1][2], b[m], low[m]);
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) low[m] = W::mfma(xt[s & 1][1], b[m], low[m]);
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) blk[m] = W::mfma(xt[s & 1][0], b[m], blk[m]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < W::NSUB; ++m) blk[m] += low[m];
        if (big) {
            // the factor goes to the scale where that is at most 1, else to the sum:
            // neither overflows unless the term does
#pragma unroll
            for (int i = 0; i < W::NV; ++i) {
                const float f = sh.f[kh * MR + W::row(lane, i)];
#pragma unroll
                for (int m = 0; m < W::NSUB; ++m) {
                    const float s = sc[m * MR / 32];
                    if (s <= 1.0f) {
                        tot[m][i] = __builtin_fmaf(blk[m][i], s * f, tot[m][i]);
                        blk[m][i] = 0.0f;  // added
                    } else {
                        blk[m][i] *= f;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < W::NV; ++i)
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) tot[m][i] = __builtin_fmaf(blk[m][i], sc[m * MR / 32], tot[m][i]);
    };
#pragma unroll
    for (int m = 0; m < W::NSUB; ++m) tot[m] = V{};
    load(0);
    store();
    __syncthreads();
    for (uint32_t it = 0; it + 1 < nit; ++it) {
        load(it + 1);
        __builtin_amdgcn_sched_barrier(0);  // the requests leave before the products
        multiply(it);
        __syncthreads();
        store();
        __syncthreads();
    }
    multiply(nit - 1);
    if constexpr (KS > 1) {  // the other K groups' sums, through the weight stage
        constexpr int NE = W::NSUB * W::NV;
        static_assert(WN * (KS - 1) * 64 * NE * 4 <= (int)sizeof(sh.w), "partial sums fit");
        __syncthreads();
        float *part = reinterpret_cast<float *>(&sh.w[0][0]) + lane;
        if (kh)
#pragma unroll
            for (int k = 0; k < NE; ++k) part[((kh - 1) * WN + wn) * 64 * NE + 64 * k] = tot[k / W::NV][k % W::NV];
        __syncthreads();
        if (!kh)
#pragma unroll
            for (int g = 1; g < KS; ++g)
#pragma unroll
                for (int k = 0; k < NE; ++k)
                    tot[k / W::NV][k % W::NV] += part[((g - 1) * WN + wn) * 64 * NE + 64 * k];
    }
}

// y_m[S][O_m] = x[S][I] . dequant(W_m)^T, I % 128 == 0: MR rows x 64 WN
// columns per workgroup.  Item t of the launch is column tile t / mtiles, row
// tile t % mtiles; each XCD (block % 8) walks a contiguous range, so a column
// tile's weights are read into one XCD's L2 once.
template <int MR, int WN, int KS>
__global__ __launch_bounds__(64 * WN * KS, 2) void k_gemm_f32x(GemvMulti G, const float *__restrict__ x, uint32_t S,
                                                                  uint32_t I) {
    __shared__ __align__(16) GFLds<MR, WN, KS> sh;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t mtiles = (S + MR - 1) / MR, T = G.blk0[G.n] * mtiles, per = (T + 7) / 8;
    const uint32_t t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || t >= T) return;  // block-uniform
    const uint32_t ct = t / mtiles, row0 = (t - ct * mtiles) * MR;
    uint32_t m = 0;
#pragma unroll
    for (uint32_t k = 1; k < CZ_GEMV_MULTI; ++k)
        if (k < G.n && ct >= G.blk0[k]) m = k;
    const uint32_t O = G.O[m], c0 = (ct - G.blk0[m]) * 64 * WN + (wave % WN) * 64;
    if (tid < MR) {
        sh.src[tid] = (uint64_t)min(row0 + tid, S - 1) * I;
        sh.dst[tid] = row0 + tid < S ? row0 + tid : ~0u;
    }
    __syncthreads();
    const uint8_t *wb[2];
    const float *sr[2];
    uint32_t rmax[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {  // columns past O read column O - 1 and are not stored
        const uint32_t nb = min(c0 + 32 * k, O - 1);
        wb[k] = G.w[m] + (uint64_t)nb * I;
        rmax[k] = O - 1 - nb;
        sr[k] = G.s[m] + (uint64_t)(nb / CZ_BLOCK) * (I / CZ_BLOCK);
    }
    typedef GFWave<MR> W;
    typename W::V tot[W::NSUB];
    cz_gf_tile<MR, WN, KS>(sh, x, I, wb, rmax, sr, tot);
    if (wave >= WN) return;  // the other K groups' waves
    float *y = G.y[m];
#pragma unroll
    for (int i = 0; i < W::NV; ++i) {
        const uint32_t dst = sh.dst[W::row(lane, i)];
        if (dst == ~0u) continue;
#pragma unroll
        for (int k = 0; k < W::NSUB; ++k) {
            const uint32_t c = c0 + MR * k + (lane & (MR - 1));
            if (c < O) y[(uint64_t)dst * O + c] = tot[k][i];
        }
    }
}

// Grouped GEMM of the routed experts: one M-tile (32 rows of one expert) x 256
// weight rows per workgroup.  GATEUP: a wave's two
// subtiles are the gate and up rows of the same 32 outputs, h = silu(g) u as
// f32; DOWN: 64 adjacent rows.  The shared expert's items (PS) run first in the
// same launch; items and their XCD ranges as in k_gg.  2000 tokens of a
// Qwen3-30B-A3B layer, Zipf(1.1): gate/up 434 us, down 250 us (medians of the
// kernel trace; least 366 and 209).
template <int MODE>
__global__ __launch_bounds__(256, 2) void k_gg_f32x(GroupArgs G, GGProblem PR, GGProblem PS, const float *__restrict__ aR,
                                                    const float *__restrict__ aS) {
    constexpr int MR = CZ_GG_M, WN = 4;
    typedef GFWave<MR> W;
    constexpr uint32_t NCOL = cz_gg_cols<MODE>();
    __shared__ __align__(16) GFLds<MR, WN, 1> sh;
    const uint32_t ns = PS.N ? (PS.rows_total + MR - 1) / MR * ((PS.N + NCOL - 1) / NCOL) : 0u, ns8 = (ns + 7u) & ~7u;
    const bool shared = blockIdx.x < ns8;
    if (shared && blockIdx.x >= ns) return;  // block-uniform
    const GGProblem P = shared ? PS : PR;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t ntn = (P.N + NCOL - 1) / NCOL;
    uint32_t t = blockIdx.x;
    if (!shared) {
        const uint32_t b = blockIdx.x - ns8, T = G.ntiles[0] * ntn, per = (T + 7) / 8;
        t = (b & 7) * per + (b >> 3);
        if ((b >> 3) >= per || t >= T) return;  // block-uniform
    }
    const uint32_t mt = t / ntn, nt = t - mt * ntn;
    uint32_t e = 0, row0 = mt * MR, rows = shared ? min((uint32_t)MR, P.rows_total - row0) : 0u;
    if (!shared) {
        e = G.tile_expert[mt];
        row0 = G.tile_row0[mt];
        rows = min((uint32_t)MR, G.offsets[e + 1] - row0);
    }
    if (tid < MR) {
        const uint32_t pos = row0 + min(tid, rows - 1);
        // GATEUP: the slot's token row of x; DOWN: the sorted row of h; shared: token rows in order
        const uint32_t src = (MODE == GG_GATEUP && !shared) ? G.sorted_slot[pos] / G.L.K : pos;
        sh.src[tid] = (uint64_t)src * P.Kd;
        sh.dst[tid] = tid < rows ? pos : ~0u;
    }
    __syncthreads();
    const uint64_t sl = shared ? 0 : cz_slot(G.L, e);
    const uint8_t *W0 = P.w0 + sl * P.w_stride;
    const float *S0 = P.s0 + sl * P.s_stride;
    const uint8_t *wb[2];
    const float *sr[2];
    uint32_t rmax[2], col[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const uint32_t c = nt * NCOL + (MODE == GG_GATEUP ? wave * 32u : wave * 64u + 32u * m);
        const uint32_t nb = min(c, P.N - 1);
        const bool up = MODE == GG_GATEUP && m;
        wb[m] = W0 + (up ? P.w1_off : 0) + (uint64_t)nb * P.Kd;
        rmax[m] = P.N - 1 - nb;
        sr[m] = S0 + (up ? P.s1_off : 0) + (uint64_t)(nb / CZ_BLOCK) * P.nbK;
        col[m] = c + (lane & (MR - 1));
    }
    typename W::V tot[W::NSUB];
    cz_gf_tile<MR, WN, 1>(sh, shared ? aS : aR, P.Kd, wb, rmax, sr, tot);
    constexpr int HS = W::NSUB / 2;  // subtiles of each 32-row half
#pragma unroll
    for (int i = 0; i < W::NV; ++i) {
        const uint32_t dst = sh.dst[W::row(lane, i)];
        if (dst == ~0u) continue;
        float *c = P.c + (uint64_t)dst * P.N;
#pragma unroll
        for (int k = 0; k < HS; ++k) {
            const uint32_t c0 = col[0] + MR * k, c1 = col[1] + MR * k;
            if constexpr (MODE == GG_GATEUP) {
                if (c0 < P.N) c[c0] = cz_silu_fast(tot[k][i]) * tot[HS + k][i];
            } else {
                if (c0 < P.N) c[c0] = tot[k][i];
                if (c1 < P.N) c[c1] = tot[HS + k][i];
            }
        }
    }
}
