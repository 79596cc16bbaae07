// What the DMA-staged GEMM kernels (gemm_dense.cuh, gemm_mopa.cuh) share:
// arguments, operand resources, the product instruction, the tile order and the
// output store.
#pragma once

#include "kernels.h"
#include "lds_dma.cuh"
#include "tile_store.cuh"

namespace smg {

namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

struct DArgs {
    const uint16_t *a, *b;
    StoreArgs st;        // alpha / add_dst: as StoreArgs (a graph, then alpha * old C)
    float beta, alpha;
    uint32_t rd;         // no graph: C = alpha * C + beta * A@B, one rounding
    uint32_t m, n, k;
    uint32_t brows;      // rows of B that can be read
    long lda, ldb;
    const uint16_t *col_a, *col_b;  // the compiled store's operands (EpPick)
    uint32_t act;
    float act_alpha;
};

// The operands as buffer resources from the tile's first row on: rows past the
// last read zeros (never stored), and so do the last step's chunks past K,
// whose lanes take the offset OOB.
__device__ __forceinline__ rsrc4_t dense_rsrc(const uint16_t *p, uint32_t row0, uint32_t rows, long ld, uint32_t k) {
    const uint64_t bytes = ((uint64_t)(rows - 1 - row0) * ld + k) * 2;
    return make_rsrc4(p + (size_t)row0 * ld, (uint32_t)(bytes < OOB ? bytes : OOB));
}

template <bool BF16>
__device__ __forceinline__ float4_t mfma16(const u32x4_t &a, const u32x4_t &b, float4_t c) {
    if (!BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b),
                                                      c, 0, 0, 0);
    } else {
        typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
}

// Output tile (tm, tn) of workgroup b: an XCD's workgroups take a contiguous
// run of tiles (xcd_tile), walked in bands of GM row tiles, so that the run
// covers a compact block and its row and column panels stay in that XCD's L2.
template <uint32_t GM>
__device__ __forceinline__ void dense_tile(uint32_t b, uint32_t grid, uint32_t mt, uint32_t nt, uint32_t &tm,
                                           uint32_t &tn) {
    const uint32_t l = xcd_tile(b, grid), band = l / (GM * nt), r0 = band * GM, in = l - r0 * nt;
    const uint32_t rows = min(GM, mt - r0);
    tm = r0 + in % rows;
    tn = in / rows;
}

// One 64-column group's staged output rows to C (rows rl0 + rstep j of R, 8
// columns cl ..), through the op-graph.
template <bool BF16, int EPV, int TBM, int TBN, int R>
__device__ __forceinline__ void dense_store(const DArgs &g, const EpArgs &ep, const EpCols &cv, const float *colv,
                                            const float *rowv, const uint16_t *tile, int cs, int rl0, int rstep,
                                            int cl, uint32_t row0, uint32_t col0) {
    if constexpr (EPV == 0) {
        if (g.st.add_dst) {
#pragma unroll 1
            for (int j = 0; j < R; j++) {
                const int rl = rl0 + rstep * j;
                ep_store8<BF16, TBM, TBN>(g.st, ep, colv, rowv, *(const uint4 *)(tile + rl * cs + cl), rl, cl, row0,
                                          col0);
            }
            return;
        }
        ep_store_rows<BF16, TBM, TBN, R>(g.st, ep, colv, rowv, tile, cs, rl0, rstep, cl, row0, col0);
    } else {
        ep_store_rows_c<BF16, R, EPV>(g.st, g.act, g.act_alpha, cv, tile, cs, rl0, rstep, cl, row0, col0);
    }
}

// Rows of the old C into the staging tile (8 columns a thread, zero outside
// C), for alpha * C + beta * acc with one rounding.
template <bool BF16, int R>
__device__ __forceinline__ void dense_load_c(const DArgs &g, uint16_t *tile, int cs, int rl0, int rstep, int cl,
                                             uint32_t row0, uint32_t col0) {
    const uint32_t col = col0 + cl;
#pragma unroll
    for (int j = 0; j < R; j++) {
        const uint32_t row = row0 + rl0 + rstep * j;
        uint32_t w4[4] = {0, 0, 0, 0};
        if (row < g.m && col < g.n) {
            const uint16_t *dp = g.st.dst + (size_t)row * g.st.dst_rs + (size_t)col * g.st.dst_cs;
            if (g.st.dst_cs == 1 && col + 8 <= g.n && ((uintptr_t)dp & 15) == 0) {
                const uint4 x = *(const uint4 *)dp;
                w4[0] = x.x;
                w4[1] = x.y;
                w4[2] = x.z;
                w4[3] = x.w;
            } else {
                const uint32_t ne = min(g.n - col, 8u);
                for (uint32_t e = 0; e < ne; e++)
                    w4[e / 2] |= (uint32_t)dp[(size_t)e * g.st.dst_cs] << (16 * (e % 2));
            }
        }
        *(uint4 *)(tile + (rl0 + rstep * j) * cs + cl) = make_uint4(w4[0], w4[1], w4[2], w4[3]);
    }
}

// Four accumulators (consecutive columns of one row) rounded into the staged
// tile; with rd the staged old C joins before the one rounding.
template <bool BF16>
__device__ __forceinline__ void dense_stage4(const DArgs &g, const float4_t &acc, uint16_t *p) {
    float x[4];
#pragma unroll
    for (int v = 0; v < 4; v++) x[v] = 0.0f + g.beta * acc[v];
    if (g.rd) {
        const u32x2_t o = *(const u32x2_t *)p;
#pragma unroll
        for (int v = 0; v < 4; v++) x[v] = g.alpha * to_f32<BF16>((uint16_t)(o[v / 2] >> (16 * (v % 2)))) + g.beta * acc[v];
    }
    const u32x2_t h = {(uint32_t)from_f32<BF16>(x[0]) | ((uint32_t)from_f32<BF16>(x[1]) << 16),
                       (uint32_t)from_f32<BF16>(x[2]) | ((uint32_t)from_f32<BF16>(x[3]) << 16)};
    *(u32x2_t *)p = h;
}

}  // namespace

}  // namespace smg
