// cz_gemm.h - E4M3 weights times f32 rows on the f16 matrix cores at f32's
// accuracy: many-token projections (matmulFp8, fp8.zig:215-257) and the
// grouped expert products of prompts past the FP8 form's slots.
//
// A K block of a row (128 columns, one weight scale block) is multiplied by a
// power of two that puts its largest element in [2^14, 2^15), then split as
// f16 hi + lo: hi keeps 11 bits, lo the next 11, so at most the last bit of an
// f32 is rounded, and elements down to 2^-16 of the largest keep all of it (no
// f16 subnormals).  E4M3 is exact in f16, every product is exact in f32, and
// each K block's sum is taken alone and then added as tot = fma(blk 2^e, s,
// tot) with the block scale s (the product with 2^e is exact).
//
// The split is done as the rows are staged in LDS, so no pass before the
// product and no scratch is needed, and the f32 row is as many bytes as hi and
// lo together.
//
// Bound: one K block of a 32 x 256 tile is 1,024 cycles of MFMA a SIMD beside
// about as many of vector work (the split, E4M3 to f16, the fold into tot) and
// of LDS traffic; two workgroups on a CU overlap them to about 3,200 cycles,
// one alone takes 4,000.  Measured and not kept: loads two K blocks ahead (the
// same time: the loads are not what is waited for), 64-row tiles with eight
// waves (1500 tokens' q, k, v 103-172 against 84 us).
#pragma once

#include "cz_grouped.h"

#define CZ_GF_ALD 272  // LDS bytes per staged K block of a row (256 + 16: rows in distinct bank groups)

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
    __device__ static __forceinline__ V mfma(cz_half8 a, cz_half8 b, V c) {
        if constexpr (MR == 32)
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// One workgroup's tile: its WN x KS waves take the same MR rows and 64 weight
// rows each; KS wave groups take every KS-th K block and their sums are added
// at the end.
template <int MR, int WN, int KS>
struct GFLds {
    static constexpr int RB = MR * KS;  // K blocks of rows staged per pass
    uint8_t hi[RB * CZ_GF_ALD];
    uint8_t lo[RB * CZ_GF_ALD];
    uint8_t w[WN * KS][64 * CZ_GG_WLD];
    float f[RB];       // 2^e that undoes each row block's scaling
    uint64_t src[MR];  // element offset of each tile row's A row
    uint32_t dst[MR];  // C row, ~0u: padding
};

// tot = the wave's products: weight rows 0-31 are wb[0]'s, 32-63 wb[1]'s (each
// clamped at rmax, scales sr); valid in the kh = 0 waves.
template <int MR, int WN, int KS>
__device__ __forceinline__ void cz_gf_tile(GFLds<MR, WN, KS> &sh, const float *__restrict__ a, uint32_t Kd,
                                           const uint8_t *const (&wb)[2], const uint32_t (&rmax)[2],
                                           const float *const (&sr)[2],
                                           typename GFWave<MR>::V (&tot)[GFWave<MR>::NSUB]) {
    typedef GFWave<MR> W;
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
        float mx[NA];
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            const float *v = (const float *)av[p];
            mx[p] = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) mx[p] = fmaxf(mx[p], __builtin_fabsf(v[i]));
        }
#pragma unroll
        for (int p = 0; p < NA; ++p) mx[p] = fmaxf(mx[p], cz_dpp<0xB1>(mx[p]));
#pragma unroll
        for (int p = 0; p < NA; ++p) mx[p] = fmaxf(mx[p], cz_dpp<0x4E>(mx[p]));
#pragma unroll
        for (int p = 0; p < NA; ++p) mx[p] = fmaxf(mx[p], cz_dpp<0x141>(mx[p]));
#pragma unroll
        for (int p = 0; p < NA; ++p) mx[p] = fmaxf(mx[p], cz_dpp<0x140>(mx[p]));
        bool inf = false;
        cz_half4 h[NA][2], l[NA][2];
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            // 2^(141 - E) and its inverse, E the biased exponent (at least 15, so
            // that both are normal); an infinity (E = 255) scales the rest down too
            const uint32_t E = max(__builtin_bit_cast(uint32_t, mx[p]) >> 23, 15u);
            const float up = __builtin_bit_cast(float, (268u - E) << 23);
            if (q == 0) sh.f[(tid >> 4) + p * (NT / 16)] = __builtin_bit_cast(float, (E - 14u) << 23);
            inf |= E == 255u;
            const float *v = (const float *)av[p];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const _Float16 hi = (_Float16)(v[i] * up);
                h[p][i / 4][i % 4] = hi;
                l[p][i / 4][i % 4] = (_Float16)__builtin_fmaf(v[i], up, -(float)hi);  // exact, then rounded
            }
        }
        if (inf) {  // inf - inf: an infinity has no lower part
#pragma unroll
            for (int p = 0; p < NA; ++p)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (__builtin_isinf(((const float *)av[p])[i])) l[p][i / 4][i % 4] = (_Float16)0.0f;
        }
#pragma unroll
        for (int p = 0; p < NA; ++p)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t o = ((tid >> 4) + p * (NT / 16)) * CZ_GF_ALD + 8 * q + 128 * i;
                *(cz_half4 *)(sh.hi + o) = h[p][i];
                *(cz_half4 *)(sh.lo + o) = l[p][i];
            }
    };
    const uint32_t rl = lane & (MR - 1), kg = lane / MR;
    const uint32_t ao = (kh * MR + rl) * CZ_GF_ALD + kg * (256 / W::G);  // + 16 s
    const uint8_t *lr = lw + rl * CZ_GG_WLD + kg * (128 / W::G);         // + 8 s: the same K order
    auto multiply = [&](uint32_t it) {
        const uint32_t kb = it * KS + kh;
        if (KS > 1 && kb >= nkb) return;  // wave-uniform
        const float sc[2] = {cz_const_f32(sr[0] + kb), cz_const_f32(sr[1] + kb)};
        V blk[W::NSUB] = {}, low[W::NSUB] = {};
        u32x4 wq[2][W::NSUB];
        cz_half8 xh[2], xl[2];
        auto fetch_w = [&](int s2) {
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) wq[s2 & 1][m] = *(const u32x4 *)(lr + m * MR * CZ_GG_WLD + 16 * s2);
        };
        auto fetch_a = [&](int s) {
            xh[s & 1] = *(const cz_half8 *)(sh.hi + ao + 16 * s);
            xl[s & 1] = *(const cz_half8 *)(sh.lo + ao + 16 * s);
        };
        fetch_w(0);
        fetch_a(0);
        fetch_w(1);
#pragma unroll
        for (int s = 0; s < W::NS; ++s) {  // step s + 1's operands are read while step s multiplies
            if (s + 1 < W::NS) fetch_a(s + 1);
            if (s >= 2 && s % 2 == 0 && s / 2 + 1 < W::NS / 2) fetch_w(s / 2 + 1);
            cz_half8 b[W::NSUB];
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) {
                const u32x4 w = wq[(s >> 1) & 1][m];
                b[m] = (s & 1) ? cz_fp8x8_to_f16(w[2], w[3]) : cz_fp8x8_to_f16(w[0], w[1]);
            }
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m)
                if constexpr (KS == 1)
                    low[m] = W::mfma(xl[s & 1], b[m], low[m]);
                else
                    blk[m] = W::mfma(xl[s & 1], b[m], blk[m]);
#pragma unroll
            for (int m = 0; m < W::NSUB; ++m) blk[m] = W::mfma(xh[s & 1], b[m], blk[m]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 0; m < W::NSUB; ++m)
            if constexpr (KS == 1) blk[m] += low[m];  // the low parts' sum is rounded into the rest once
#pragma unroll
        for (int j = 0; j < W::NV / 4; ++j) {
            const float4 f4 = *(const float4 *)(sh.f + kh * MR + W::row(lane, 4 * j));
            const float f[4] = {f4.x, f4.y, f4.z, f4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int m = 0; m < W::NSUB; ++m)
                    tot[m][4 * j + i] = __builtin_fmaf(blk[m][4 * j + i] * f[i], sc[m * MR / 32], tot[m][4 * j + i]);
        }
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
// tile's weights are read into one XCD's L2 once.  Error against 64 bits at the
// Qwen3-30B-A3B projections 1.2-1.3e-7 (the GEMV's: 1.6e-7).
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
// Qwen3-30B-A3B layer, Zipf(1.1): gate/up 313 us, down 177 us; the layer's
// error against 64 bits 2.4e-7 (the per-token kernels': 2.6e-7).
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
