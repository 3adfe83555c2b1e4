// cz_native.h - BF16 rows on several tokens through the f32 matrix cores, every
// dot in dotBf16's order (matmul.zig:84-110) bit for bit.
//
// v_mfma_f32_4x4x1_16b_f32 is 16 independent 4 x 4 outer products, each
// D[i][j] = fma(A[i], B[j], C[i][j]): one FMA per element and no sum inside the
// instruction (checked on the device over 2^22 operands, every bit pattern
// class, denormals and NaN payloads included).  So a chain of them is a chain
// of FMAs, and an accumulator that takes one of dotBf16's 32 chains keeps that
// chain's order.
#pragma once

#include "cz_kernels.h"

typedef float cz_float4v __attribute__((ext_vector_type(4)));

// y[S][O] = x[S][I] . W^T, W BF16 [O][I], I % 256 == 0.
//
// A wave takes 16 rows and 4 TG tokens; TH = 2: the workgroup's second four
// waves take its other 4 TG tokens on the same rows (their weight reads hit
// the caches), because accumulators for 16 tokens leave one wave a SIMD.  Block b of an MFMA is
// row quad b / 4 and chain group b % 4; lane l gives A = row 4 (l / 16) + l % 4
// and B = token l % 4, both at chain group (l / 4) % 4.  A lane's 16-byte load
// is the 8 chains 8 (b % 4) + e of its row at one 32-wide step, so accumulator
// e of the lane's block runs chain 8 (b % 4) + e through every step.  After the
// last step the four chain groups of a row quad, 4 lanes apart, are added in
// dotBf16's order, then the 8 lanes of the reference's vector, which are the
// accumulators e.
//
// The workgroup's tokens stay in LDS for all its rows, in the order the B
// operand reads them ([step][token group][half][chain group][token] of 16
// bytes: a 16-lane read is 256 contiguous bytes, the four row quads broadcast).
//
// Bound: HBM reads of W (622 MB at 151936 x 2048: 101 us at one token's
// measured 6.1 TB/s), then the matrix cores and LDS, 16 us per four tokens
// each.  151936 x 2048 rows, the row kernel before and now: 2 tokens 129 and
// 117 us, 4 169 and 120, 8 262 and 130 (4.8 TB/s), 12 405 and 155, 16 490 and 231.
// More or fewer loads in flight (4 or 16 steps a block), non-temporal loads and
// staggered waves measured the same or slower.
template <int TG, int TH>
__global__ __launch_bounds__(512, 2) void k_native_mfma(float *__restrict__ y, const float *__restrict__ x,
                                                        const uint16_t *__restrict__ w, uint32_t S, uint32_t I,
                                                        uint32_t O) {
    constexpr int U = TG <= 2 ? 8 : 4;  // steps per block of loads (16 bytes a lane each)
    constexpr int NSET = 3;  // register sets: two blocks in flight while one is multiplied
    constexpr uint32_t TW = TG * TH, NWV = 8 / TH;  // token groups and row tiles of the workgroup
    extern __shared__ float4 cz_native_xs[];
    float4 *xs = cz_native_xs;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t g0 = wave / NWV * TG;  // the wave's first token group
    const uint32_t t0 = blockIdx.y * 4 * TW, I4 = I / 4, nb = I / (32 * U);
    const uint32_t tiles = (O + 15) / 16, stride = gridDim.x * NWV;
    const uint32_t arow = (lane >> 4) * 4 + (lane & 3), cg = (lane >> 2) & 3;
    // the wave's blocks in order, tile after tile: loads run ahead across the
    // end of a tile (past the last tile row O - 1 is read again, unused)
    uint32_t tile = blockIdx.x * NWV + wave % NWV, blk = 0, ltile = tile, lblk = 0;
    auto row = [&](uint32_t t) { return w + (uint64_t)min(t * 16 + arow, O - 1) * I + cg * 8; };
    const uint16_t *lp = row(ltile);
    auto load = [&](uint4(&d)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) d[u] = *(const uint4 *)(lp + 32 * u);
        __builtin_amdgcn_sched_barrier(0);  // the requests leave before the products of the block in hand
        lp += 32 * U;
        if (++lblk == nb) {
            lblk = 0;
            ltile += stride;
            lp = row(ltile);
        }
    };
    uint4 a[NSET][U];
#pragma unroll
    for (int k = 0; k < NSET - 1; ++k) load(a[k]);
    for (uint32_t i = tid; i < 4 * TW * I4; i += 512) {
        const uint32_t t = i / I4, c = i - t * I4;  // 16-byte chunk c of token t0 + t
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (t0 + t < S) v = reinterpret_cast<const float4 *>(x)[(uint64_t)(t0 + t) * I4 + c];
        xs[(((c >> 3) * TW + (t >> 2)) * 2 + (c & 1)) * 16 + ((c >> 1) & 3) * 4 + (t & 3)] = v;
    }
    __syncthreads();
    if (tile >= tiles) return;  // wave-uniform, past the only barrier
    cz_float4v acc[8][TG];
    auto clear = [&] {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int g = 0; g < TG; ++g) acc[e][g] = cz_float4v{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    // one block: request the next one into nxt, multiply cur; true after the
    // wave's last tile
    auto step = [&](const uint4(&cur)[U], uint4(&nxt)[U]) -> bool {
        load(nxt);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t q[4] = {cur[u].x, cur[u].y, cur[u].z, cur[u].w};
            float b[TG][8];
#pragma unroll
            for (int g = 0; g < TG; ++g)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *(float4 *)&b[g][4 * h] = xs[(((blk * U + u) * TW + g0 + g) * 2 + h) * 16 + (lane & 15)];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float av = __builtin_bit_cast(float, (e & 1) ? q[e / 2] & 0xffff0000u : q[e / 2] << 16);
#pragma unroll
                for (int g = 0; g < TG; ++g)
                    acc[e][g] = __builtin_amdgcn_mfma_f32_4x4x1f32(av, b[g][e], acc[e][g], 0, 0, 0);
            }
            if constexpr (TG >= 3) __builtin_amdgcn_sched_barrier(0);  // one step's operands at a time in registers
        }
        if (++blk < nb) return false;
        // (((0 + g0) + g1) + g2) + g3 over the chain groups in the lanes of
        // group 0, then the eight lanes from -0
#pragma unroll
        for (int g = 0; g < TG; ++g) {
            const uint32_t t = t0 + 4 * (g0 + g) + (lane & 3), r0 = tile * 16 + (lane >> 4) * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float sum = -0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float v = acc[e][g][i];
                    float c = 0.0f + v;
                    c = c + cz_dpp<0x104>(v);  // row_shl:4
                    c = c + cz_dpp<0x108>(v);
                    c = c + cz_dpp<0x10C>(v);
                    sum = sum + c;
                }
                if (cg == 0 && t < S && r0 + i < O) y[(uint64_t)t * O + r0 + i] = sum;
            }
        }
        clear();
        blk = 0;
        tile += stride;
        return tile >= tiles;
    };
    for (;;) {
        if (step(a[0], a[2])) return;
        if (step(a[1], a[0])) return;
        if (step(a[2], a[1])) return;
    }
}
