// Many-row 2-bit / 1-bit int8 products: matmul_q2 / matmul_q1 (+ _ep) past the
// decode kernels' rows (prefill), bit for bit the portable path
// (src/kernels/lowbit/matmul.rs:354-398), replacing the panel loop of
// csrc/gemm_q2.cc:48-429 there.
//
// lowbit_quant_frag quantizes A once, a wave per (16 rows, block), straight
//   into the order the products read: the 16 bytes lane l of
//   v_mfma_i32_16x16x64_i8's B operand holds (row l % 16, depths 16 (l / 16)
//   of the slab) at byte 16 l of the (row tile, slab)'s 1 KB, so a wave's
//   fragment is one contiguous, conflict-free LDS read and a tile's DMA is
//   linear.
// lowbit_gemm: a workgroup of 4 waves owns 16 RT rows x 64 CT columns, a wave
//   16 CT of the columns. Everything a 256-depth step needs -- the rows'
//   fragments, the columns' codes, their scales and the rows' block scales --
//   goes global -> LDS by DMA, NSTG - 1 steps ahead. Codes are expanded to
//   int8 in registers once per 16 RT rows (v_perm_b32 with the codebook as the
//   table; Q1 is the codebook {-1, +1}), a block's products accumulate from
//   zero in i32 (exact), and each block folds at once into the f32 totals the
//   lanes keep, total = fmaf(f32(sum), f32(scale) * s, total), in block order
//   as the reference does. A row tile's fold runs beside the next row tile's
//   products.
// What bounds it: the fold's three vector instructions an output and block
//   (convert, scale product, fma) and the expansion, about twice the matrix
//   cores' time for the same block (2-bit 512 x 11008 x 4096: vector issue 57 % of
//   the kernel's cycles, products 19 %); so the expansion is shared by RT row
//   tiles and several waves a SIMD overlap one's fold with another's
//   products.
#include <algorithm>

#include "kernels.h"
#include "lds_dma.cuh"

namespace smg {

namespace {

constexpr int LG_NT = 256;         // threads
constexpr uint32_t LG_STEP = 256;  // depths a step (4 slabs)

struct LgArgs {
    const uint8_t *codes;
    const uint16_t *sc;
    uint16_t *dst;
    const int8_t *q;  // [mt16][nsteps * 4 slabs][64 lanes][16]
    const float *s;   // [nsteps * blocks a step][16 mt16]
    uint32_t m, n, n_pad;
    uint32_t nsteps, nbk;   // 256-depth steps, blocks that hold depths below k
    uint32_t mt16;          // 16-row tiles of A
    uint32_t codebook;
    // the compiled store's operands (EpPick's a, b, act, alpha)
    const uint16_t *col_a, *col_b;
    uint32_t act;
    float act_alpha;
};

// A wave per (16 rows, block of SPB slabs): amax, inv, s and q as quantize_row
// (src/kernels/lowbit/matmul.rs:354-371). Rows past m and depths past k are
// zero. The packed-u16 maximum of |a|'s bits orders as the values do, with NaN
// above infinity, so a NaN anywhere makes amax NaN as the reference's does.
// VEC: rows of whole, 16-byte-aligned groups of 8. Other rows are read 64
// consecutive depths a wave's load and turned through LDS: a lane's own 16 depths
// read element by element touched 64 places a load, and took a call of few rows
// and columns up to 3 us longer (2-bit 64 x 700 x 2001, blocks of 256).
template <int SPB, bool VEC>
__global__ void __launch_bounds__(256) lowbit_quant_frag(const uint16_t *lhs, uint32_t m, uint32_t k, uint32_t nslab,
                                                         uint32_t mt16, uint32_t nbk, int8_t *q, float *s) {
    const uint32_t w = blockIdx.x * 4 + threadIdx.x / 64;
    if (w >= mt16 * nbk) return;  // whole waves, no barrier follows
    const uint32_t mt = w % mt16, blk = w / mt16;
    const int lane = threadIdx.x % 64, gq = lane / 16, c = lane % 16;
    const uint32_t row = mt * 16 + c;
    const rsrc_t ar = make_rsrc(lhs, m * k * 2u);
    uint4 a[SPB][2];
    if constexpr (VEC) {
#pragma unroll
        for (int u = 0; u < SPB; u++) {
            const uint32_t d = (blk * SPB + u) * LB_SLAB + 16 * gq;
            a[u][0] = load_row8(ar, row, m, k, d, true);
            a[u][1] = load_row8(ar, row, m, k, d + 8, true);
        }
    } else {
        constexpr int RS = SPB * LB_SLAB + 8;  // halfs a staged row
        __shared__ __align__(16) uint16_t rows[4][16 * RS];
        uint16_t *st = rows[threadIdx.x / 64];  // the wave's own
        uint16_t e[16][SPB];
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
            for (int u = 0; u < SPB; u++) {
                const uint32_t rr = mt * 16 + r, d = (blk * SPB + u) * LB_SLAB + lane;
                e[r][u] = bload2(ar, rr < m && d < k ? (rr * k + d) * 2u : OOB);
            }
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
            for (int u = 0; u < SPB; u++) st[r * RS + u * LB_SLAB + lane] = e[r][u];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int u = 0; u < SPB; u++)
#pragma unroll
            for (int h = 0; h < 2; h++) a[u][h] = *(const uint4 *)(st + c * RS + u * LB_SLAB + 16 * gq + 8 * h);
    }
    uint32_t mx = 0;
#pragma unroll
    for (int u = 0; u < SPB; u++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t w4[4] = {a[u][h].x, a[u][h].y, a[u][h].z, a[u][h].w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t b = w4[e] & 0x7FFF7FFFu;
                mx = max(mx, max(b & 0xFFFFu, b >> 16));
            }
        }
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, 16));
    mx = max(mx, (uint32_t)__shfl_xor((int)mx, 32));
    const float amax = f16_to_f32((uint16_t)mx);
    const float inv = amax > 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
#pragma unroll
    for (int u = 0; u < SPB; u++) {
        uint4 o;
        o.x = quant4(a[u][0].x, a[u][0].y, inv);
        o.y = quant4(a[u][0].z, a[u][0].w, inv);
        o.z = quant4(a[u][1].x, a[u][1].y, inv);
        o.w = quant4(a[u][1].z, a[u][1].w, inv);
        *(uint4 *)(q + (((size_t)mt * nslab + blk * SPB + u) * 64 + lane) * 16) = o;
    }
    if (gq == 0) s[(size_t)blk * mt16 * 16 + row] = __fdiv_rn(amax, 127.0f);
}

// f32(scale) * s with the f32 rounding of the product (the f16 scale widened
// exactly; a -0 addend leaves the product as it is).
__device__ __forceinline__ float scale_mul_lo(uint32_t sc2, float s) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(sc2), "v"(s), "v"(-0.0f));
    return r;
}
__device__ __forceinline__ float scale_mul_hi(uint32_t sc2, float s) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(sc2), "v"(s), "v"(-0.0f));
    return r;
}

// Four cells' activation with the kind switch taken once, the f64 formulas as
// act_f32 evaluates them.
struct F4 {
    float v[4];
};
__device__ __noinline__ F4 act4(uint32_t kind, F4 x, float alpha) {
    const double a = (double)alpha;
    switch (kind) {
#define SMG_ACT4_CASE(K)                                                                                   \
    case K:                                                                                                \
        _Pragma("unroll") for (int e = 0; e < 4; e++) x.v[e] = (float)act_f64_body(K, (double)x.v[e], a);  \
        break;
        SMG_ACT4_CASE(1) SMG_ACT4_CASE(2) SMG_ACT4_CASE(3) SMG_ACT4_CASE(4) SMG_ACT4_CASE(5)
        SMG_ACT4_CASE(6) SMG_ACT4_CASE(7) SMG_ACT4_CASE(8) SMG_ACT4_CASE(9) SMG_ACT4_CASE(10)
        SMG_ACT4_CASE(11) SMG_ACT4_CASE(12) SMG_ACT4_CASE(13) SMG_ACT4_CASE(14)
        SMG_ACT4_CASE(15) SMG_ACT4_CASE(16) SMG_ACT4_CASE(17) SMG_ACT4_CASE(18)
        SMG_ACT4_CASE(19) SMG_ACT4_CASE(20) SMG_ACT4_CASE(21) SMG_ACT4_CASE(22)
        SMG_ACT4_CASE(23) SMG_ACT4_CASE(24)
#undef SMG_ACT4_CASE
    default:
        break;
    }
    return x;
}

// Four cells' last activation, rounded: act_round16 four at a time.
__device__ __forceinline__ void act_round4(uint32_t kind, const float (&x)[4], float alpha, uint16_t (&h)[4]) {
    if (kind == EP_ACT_SILU || kind == EP_ACT_SIGMOID) {  // mostly without the f64 formula
#pragma unroll
        for (int j = 0; j < 4; j++) h[j] = act_round16<false>(kind, x[j], alpha);
        return;
    }
    const F4 y = act4(kind, F4{{x[0], x[1], x[2], x[3]}}, alpha);
#pragma unroll
    for (int j = 0; j < 4; j++) h[j] = f32_to_f16(y.v[j]);
}

// ep_cell for four cells of a column side by side, each node's operands loaded
// together; a row past the output reads the last one's.
__device__ __forceinline__ void ep_cells4(const EpArgs &ep, float (&x)[4], const uint32_t (&row)[4], uint32_t col,
                                          uint32_t m, uint32_t n, uint16_t (&h)[4]) {
    for (uint32_t t = 0; t < ep.n_nodes; t++) {
        const EpNode &nd = ep.nodes[t];
        const uint16_t *p = (const uint16_t *)nd.ptr;
        if (ep.fam[t] == EPF_ACT) {
            if (t + 1 == ep.n_nodes) {
                act_round4(nd.aux, x, nd.scalar, h);
                return;
            }
            const F4 y = act4(nd.aux, F4{{x[0], x[1], x[2], x[3]}}, nd.scalar);
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = y.v[j];
            continue;
        }
        const uint32_t cls = ep.cls[t];
        const size_t ld = nd.ld == 0 ? n : nd.ld;
        if (cls == EPC_ROW || cls == EPC_TENSOR) {
            uint16_t raw[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const size_t r = min(row[j], m - 1);
                raw[j] = p[cls == EPC_ROW ? r : r * ld + col];
            }
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = ep_arith(ep.fam[t], x[j], f16_to_f32(raw[j]));
        } else {
            const float v = cls == EPC_COL ? f16_to_f32(p[col]) : nd.scalar;
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = ep_arith(ep.fam[t], x[j], v);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) h[j] = f32_to_f16(x[j]);
}

// LDS bytes of a stage: row fragments, codes, scales and row scales (a block's
// columns and rows each take one dword DMA of a wave, 256 bytes).
template <int KIND, int SPB, int RT, int CT>
struct LgStage {
    static constexpr int NB = 4 / SPB;
    static constexpr int CODES = KIND == 2 ? 1024 : 512;  // a column tile's
    static constexpr int A = 0, W = RT * 4096, SC = W + 4 * CT * CODES, S = SC + NB * 256, BYTES = S + NB * 256;
    static constexpr int PS = RT + CT * (KIND == 2 ? 1 : 2) + 2;  // DMA instructions a wave
};

// SPB: slabs a block (1, 2 or 4: blocks of 64, 128 or 256). EPV: 0 the
// interpreted graph, 1 none, 2 [mul_col] [add_col] + act (pick_ep's 2 and 3).
// (At least two waves a SIMD, so at most 256 registers: the accumulators then
// are vector registers, which the fold reads directly.)
template <int KIND, int SPB, int RT, int CT, int NSTG, int EPV>
__global__ void __launch_bounds__(LG_NT, 2) lowbit_gemm(LgArgs g, EpArgs ep) {
    using ST = LgStage<KIND, SPB, RT, CT>;
    constexpr int NB = ST::NB, TN = 64 * CT, CS = TN + 8;  // tile columns; halfs per staged output row
    constexpr int TILE = RT * 16 * CS * 2;
    __shared__ __align__(16) uint8_t smem[NSTG * ST::BYTES > TILE ? NSTG * ST::BYTES : TILE];

    const uint32_t mtiles = (g.mt16 + RT - 1) / RT;
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);  // consecutive workgroups share codes
    const uint32_t rt0 = (tile % mtiles) * RT, col0 = (tile / mtiles) * TN;
    const int t = threadIdx.x, lane = t % 64, gq = lane / 16, c = lane % 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const uint32_t lds0 = lds_addr(smem);
    const uint32_t nslab = g.nsteps * 4, mld = g.mt16 * 16, last = g.nsteps - 1;
    const uint32_t kb = wave % NB;  // the block whose scales this wave loads

    // per-lane source offsets: codes (cell of column lane % 16, quarter lane /
    // 16), the scales' column pair, the row scale (rows past A's row tiles
    // repeat its last one; columns past the tile's half a wave repeat)
    uint32_t off_w[CT];
#pragma unroll
    for (int i = 0; i < CT; i++)
        off_w[i] = (uint32_t)cell_col_part(col0 + (wave * CT + i) * 16 + c, 0, g.n_pad) * 64 + gq * 16;
    const uint32_t off_sc = (uint32_t)cell_col_part(col0 + (2 * lane) % TN, 0, g.n_pad) * 2;
    const uint32_t off_s = min(rt0 * 16 + lane % (RT * 16), mld - 1) * 4;
    auto dma = [&](uint32_t step, uint32_t stage) {
        const uint32_t ks = min(step, last), base = lds0 + stage * ST::BYTES;
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int p = wave * RT + i;  // piece: row tile p / 4, slab p % 4
            const uint32_t rt = min(rt0 + p / 4, g.mt16 - 1);
            dma16(g.q + ((size_t)rt * nslab + ks * 4 + p % 4) * 1024, lane * 16, base + p * 1024);
        }
        const uint8_t *cp = g.codes + cell_row_part(KIND == 2 ? ks : ks / 2, 0, g.n_pad) * 64;
#pragma unroll
        for (int i = 0; i < CT; i++) {
            const uint32_t dst = base + ST::W + (wave * CT + i) * ST::CODES;
            if (KIND == 2) {
                dma16(cp, off_w[i], dst);
            } else {  // the step's half of a group: two dwords a lane
                dma4(cp + (ks & 1) * 8, off_w[i], dst);
                dma4(cp + (ks & 1) * 8 + 4, off_w[i], dst + 256);
            }
        }
        const uint32_t blk = ks * NB + kb;
        dma4(g.sc + cell_row_part(blk, 0, g.n_pad), off_sc, base + ST::SC + kb * 256);
        dma4(g.s + (size_t)blk * mld, off_s, base + ST::S + kb * 256);
    };

    float4_t total[CT][RT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int i = 0; i < RT; i++) total[ct][i] = (float4_t){0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int j = 0; j < NSTG - 1; j++) dma(j, j);
    const uint32_t cb = KIND == 2 ? g.codebook : 0x000001FFu;
    uint32_t stage = 0;
    for (uint32_t ks = 0; ks < g.nsteps; ks++) {
        // step ks has landed for every wave, and every wave has read step
        // ks - 1's stage for the last time
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        wait_vm<(NSTG - 2) * ST::PS>();
        barrier_lds();
        dma(ks + NSTG - 1, stage == 0 ? NSTG - 1 : stage - 1);
        const uint32_t sb = lds0 + stage * ST::BYTES;
        stage = stage + 1 == NSTG ? 0 : stage + 1;
        uint32_t w[CT][4];
        uint2 sc[NB][CT];
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            const uint32_t wp = sb + ST::W + (wave * CT + ct) * ST::CODES;
            if (KIND == 2) {
                const int4_t x = lds_load<int4_t>(wp + lane * 16);
#pragma unroll
                for (int u = 0; u < 4; u++) w[ct][u] = (uint32_t)x[u];
            } else {
                w[ct][0] = lds_load<uint32_t>(wp + lane * 4);
                w[ct][1] = lds_load<uint32_t>(wp + 256 + lane * 4);
            }
#pragma unroll
            for (int b = 0; b < NB; b++) {
                typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
                const u32x2_t x = lds_load<u32x2_t>(sb + ST::SC + b * 256 + ((wave * CT + ct) * 16 + 4 * gq) * 2);
                sc[b][ct] = make_uint2(x[0], x[1]);
            }
        }
        // the step's NB * RT (block, row tile) units: unit p's products are
        // issued, then unit p - 1 is folded
        int4_t acc[2][CT], af[2][SPB], wf[CT][SPB];
        float s[2];
        auto read = [&](int p) {
            const int b = p / RT, i = p % RT;
#pragma unroll
            for (int u = 0; u < SPB; u++) af[p & 1][u] = lds_load<int4_t>(sb + (i * 4 + b * SPB + u) * 1024 + lane * 16);
        };
        auto expand = [&](int b) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int u = 0; u < SPB; u++) {
                    const int sl = b * SPB + u;
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        wf[ct][u][j] =
                            KIND == 2 ? (int)__builtin_amdgcn_perm(cb, cb, (w[ct][sl] >> (2 * j)) & 0x03030303u)
                                      : (int)__builtin_amdgcn_perm(cb, cb,
                                                                   (w[ct][sl / 2] >> (4 * (sl % 2) + j)) & 0x01010101u);
                }
        };
        auto mul = [&](int p) {
            s[p & 1] = lds_load<float>(sb + ST::S + (p / RT) * 256 + ((p % RT) * 16 + c) * 4);
#pragma unroll
            for (int ct = 0; ct < CT; ct++) acc[p & 1][ct] = (int4_t){0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < SPB; u++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++)
                    acc[p & 1][ct] =
                        __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[ct][u], af[p & 1][u], acc[p & 1][ct], 0, 0, 0);
        };
        auto fold = [&](int p) {
            const int b = p / RT, i = p % RT;
            const float sv = s[p & 1];
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const float y[4] = {scale_mul_lo(sc[b][ct].x, sv), scale_mul_hi(sc[b][ct].x, sv),
                                    scale_mul_lo(sc[b][ct].y, sv), scale_mul_hi(sc[b][ct].y, sv)};
#pragma unroll
                for (int v = 0; v < 4; v++) total[ct][i][v] = fmaf((float)acc[p & 1][ct][v], y[v], total[ct][i][v]);
            }
        };
        const int nb = min((int)(g.nbk - ks * NB), NB);  // blocks past k are not folded
        read(0);
        expand(0);
        if (nb == NB) {
#pragma unroll
            for (int p = 0; p < NB * RT; p++) {
                if (p + 1 < NB * RT) read(p + 1);
                mul(p);
                if (p > 0) fold(p - 1);
                if ((p + 1) % RT == 0 && p + 1 < NB * RT) expand((p + 1) / RT);
                __builtin_amdgcn_sched_barrier(0);
            }
            fold(NB * RT - 1);
        } else {
#pragma unroll
            for (int b = 0; b < NB - 1; b++) {
                if (b >= nb) break;
                if (b > 0) expand(b);
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    if (b + i > 0) read(b * RT + i);
                    mul(b * RT + i);
                    fold(b * RT + i);
                }
            }
        }
    }
    wait_vm<0>();  // the steps issued past the last

    // Store: the f16 sums staged row-major in LDS (lane: 4 consecutive columns
    // of its row), then each thread takes groups of 8 columns of a row, or, where
    // the graph has an activation or is interpreted, four cells of a column.
    __syncthreads();
    uint16_t *stg = (uint16_t *)smem;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int i = 0; i < RT; i++) {
            uint2 h;
            h.x = (uint32_t)f32_to_f16(total[ct][i][0]) | ((uint32_t)f32_to_f16(total[ct][i][1]) << 16);
            h.y = (uint32_t)f32_to_f16(total[ct][i][2]) | ((uint32_t)f32_to_f16(total[ct][i][3]) << 16);
            *(uint2 *)(stg + (i * 16 + c) * CS + wave * CT * 16 + ct * 16 + 4 * gq) = h;
        }
    __syncthreads();
    if (EPV == 0 || (EPV == 2 && g.act != EP_ACT_NONE)) {
        // four cells of one column a thread: the graph's operand loads and the
        // f64 formulas are chains, so the cells run side by side
        static_assert(LG_NT % TN == 0, "a thread's column");
        constexpr int RS = LG_NT / TN;  // rows a pass
        const uint32_t cl = t % TN, col = col0 + cl;
        if (col >= g.n) return;  // no barrier follows
        const float va = EPV == 2 && g.col_a ? f16_to_f32(g.col_a[col]) : 1.0f;
        const float vb = EPV == 2 ? f16_to_f32(g.col_b[col]) : 0.0f;
#pragma unroll 1
        for (int rl = t / TN; rl < RT * 16; rl += 4 * RS) {
            float x[4];
            uint32_t row[4];
            uint16_t h[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                row[j] = rt0 * 16 + rl + j * RS;
                x[j] = f16_to_f32(stg[(rl + j * RS) * CS + cl]);
            }
            if constexpr (EPV == 2) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (g.col_a) x[j] = x[j] * va;
                    x[j] = x[j] + vb;
                }
                act_round4(g.act, x, g.act_alpha, h);
            } else {
                ep_cells4(ep, x, row, col, g.m, g.n, h);
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (row[j] < g.m) g.dst[(size_t)row[j] * g.n + col] = h[j];
        }
        return;
    }
    const uint32_t cl = (t % (TN / 8)) * 8, col = col0 + cl;
    if (col >= g.n) return;  // no barrier follows
    const uint32_t ne = min(g.n - col, 8u);
    float va[8], vb[8];
    if constexpr (EPV == 2) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            va[e] = g.col_a && (uint32_t)e < ne ? f16_to_f32(g.col_a[col + e]) : 1.0f;
            vb[e] = (uint32_t)e < ne ? f16_to_f32(g.col_b[col + e]) : 0.0f;
        }
    }
#pragma unroll 1
    for (int rl = t / (TN / 8); rl < RT * 16; rl += LG_NT / (TN / 8)) {
        const uint32_t row = rt0 * 16 + rl;
        if (row >= g.m) break;
        const uint4 c8 = *(const uint4 *)(stg + rl * CS + cl);
        uint32_t w4[4] = {c8.x, c8.y, c8.z, c8.w};
        if constexpr (EPV == 2) {
            uint32_t o4[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if ((uint32_t)e >= ne) break;
                float x = f16_to_f32((uint16_t)(w4[e / 2] >> (16 * (e % 2))));
                if (g.col_a) x = x * va[e];
                o4[e / 2] |= (uint32_t)f32_to_f16(x + vb[e]) << (16 * (e % 2));
            }
#pragma unroll
            for (int e = 0; e < 4; e++) w4[e] = o4[e];
        }
        uint16_t *dp = g.dst + (size_t)row * g.n + col;
        if (ne == 8 && ((uintptr_t)dp & 15) == 0) {
            *(uint4 *)dp = make_uint4(w4[0], w4[1], w4[2], w4[3]);
            continue;
        }
        for (uint32_t e = 0; e < ne; e++) dp[e] = (uint16_t)(w4[e / 2] >> (16 * (e % 2)));
    }
}

uint32_t lg_steps(const WDev &w) { return (uint32_t)((w.k + LG_STEP - 1) / LG_STEP); }
size_t lg_q_bytes(const WDev &w, size_t m) { return (m + 15) / 16 * 16 * lg_steps(w) * LG_STEP; }

template <int KIND, int SPB, int RT, int CT, int NSTG>
hipError_t launch_lg(const LgArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    const uint32_t grid = (g.mt16 + RT - 1) / RT * (g.n_pad / (64 * CT));
    if (epv == 1)
        hipLaunchKernelGGL((lowbit_gemm<KIND, SPB, RT, CT, NSTG, 1>), dim3(grid), dim3(LG_NT), 0, s, g, ep);
    else if (epv == 2)
        hipLaunchKernelGGL((lowbit_gemm<KIND, SPB, RT, CT, NSTG, 2>), dim3(grid), dim3(LG_NT), 0, s, g, ep);
    else
        hipLaunchKernelGGL((lowbit_gemm<KIND, SPB, RT, CT, NSTG, 0>), dim3(grid), dim3(LG_NT), 0, s, g, ep);
    return hipGetLastError();
}
// The tile: the smallest whose workgroups are at most 11/4 of the compute
// units. Few rows or columns run many small tiles with deep rings (a step's
// latency is what they wait for); past that a larger tile's shared expansion
// and fragment reads win. Measured on 256 compute units, K = 4096, blocks of 128
// (us, tiles of 16x64 / 32x64 / 64x64 / 64x128 rows x columns): 2-bit N = 11008 at 64
// rows 16.3 / 16.4 / 18.0 / 24.0, at 128 rows 25.2 / 20.9 / 22.6 / 25.3, at 256
// rows 39.0 / 34.9 / 34.3 / 36.6, at 512 rows 69.8 / 57.0 / 56.2 / 48.4; N =
// 4096 at 64 rows 12.2 / 14.3 / 17.5 / 23.7, at 512 rows 32.7 / 29.6 / 25.5 /
// 27.8; 1-bit N = 14336 at 512 rows 148.9 / 88.2 / 67.6 / 62.6. (The 16-row
// GEMV launches these calls took before, which read every weight once per 16
// rows: N = 11008 at 16 / 64 / 512 rows 22.1 / 59.3 / 424, here 12.0 / 16.3 /
// 46.4; N = 4096 at 9 rows 11.7, here 11.7. Blocks of 64 and 256, the same rule,
// GEMV and here: N = 5000, K = 4096 at 9 / 64 / 130 rows 18.8 / 42.4 / 84.2 and 12.5 /
// 14.0 / 19.4, 14.1 / 28.8 / 56.3 and 12.2 / 13.5 / 16.2.)
TileDims lg_tile(size_t mt16, size_t n_pad) {
    const size_t cols = n_pad / 64, most = (size_t)device_cus() * 11 / 4;
    for (uint32_t rt : {1u, 2u, 4u})
        if ((mt16 + rt - 1) / rt * cols <= most) return {16 * rt, 64};
    return {64, 128};
}
template <int KIND, int SPB>
hipError_t launch_lg_rows(const LgArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    const TileDims t = lg_tile(g.mt16, g.n_pad);
    if (t.cols == 128) return launch_lg<KIND, SPB, 4, 2, 2>(g, ep, epv, s);
    if (t.rows == 16) return launch_lg<KIND, SPB, 1, 1, 4>(g, ep, epv, s);
    if (t.rows == 32) return launch_lg<KIND, SPB, 2, 1, 4>(g, ep, epv, s);
    return launch_lg<KIND, SPB, 4, 1, 3>(g, ep, epv, s);
}

}  // namespace

// Calls the 16-row GEMV takes no longer than the GEMM: blocks of 256 (9 rows x 700
// x 8000 take the GEMV 21.8, 18.7 and 16.0 us with blocks of 64, 128 and 256, its
// folds being its longest step, the GEMM 20.4, 18.4 and 18.8) past 2048 depths, few
// rows, and GEMV workgroups (16 rows x 16 columns) that fit the
// compute units once, so that no weight is waited for twice. 2-bit, us, GEMV and
// GEMM: 9 rows x 700 x 8000 16.0 / 18.8, 32 x 2048 x 4096 12.2 / 12.5, 48 x 700 x
// 4096 12.3 / 13.0; the other side: 33 x 2048 x 8000 20.8 / 18.6 (a second round),
// 64 x 128 x 16000 33.5 / 31.1 (a row group's loads compete for longer), 9 x 700 x
// 2048 10.1 / 10.3, blocks of 128 9 x 2048 x 8000 18.5 / 18.1.
static bool lowbit_gemv_faster(const WDev &w, size_t m) {
    constexpr size_t CUS = 256;  // (a constant: scratch is sized by the same rule, on any current device)
    return w.block == 256 && w.k > 2048 && m <= (w.k <= 8192 ? 64 : 32) && (m + 15) / 16 * (w.n_pad / 16) <= CUS;
}

size_t lowbit_gemm_bytes(const WDev &w, size_t m) {
    if (m < LOWBIT_GEMM_ROWS || w.k == 0 || w.n == 0 || (w.block != 64 && w.block != 128 && w.block != 256)) return 0;
    if (lowbit_gemv_faster(w, m)) return 0;
    // the GEMV's limits (a buffer resource spans < 2 GiB), and a column's code
    // offset, 256 bytes of stride a column, in the DMA's 32-bit lane offset
    const size_t kq = (w.k + w.block - 1) / w.block * w.block;
    if (m * kq >= ((size_t)1 << 31) || m * w.k * 2 >= ((size_t)1 << 31) ||
        cell_grid_rows(w.sc_rows) * w.n_pad * 2 >= ((size_t)1 << 31) || w.n_pad * 256 >= ((size_t)1 << 31))
        return 0;
    const size_t blocks = lg_steps(w) * (LG_STEP / w.block);
    return lg_q_bytes(w, m) + blocks * ((m + 15) / 16 * 16) * sizeof(float);
}

TileDims lowbit_gemm_tile(const WDev &w, size_t m) {
    if (!lowbit_gemm_bytes(w, m)) return {0, 0};
    return lg_tile((m + 15) / 16, w.n_pad);
}

hipError_t launch_lowbit_gemm(const WDev &w, size_t m, uint16_t *dst, const uint16_t *lhs, const EpArgs &ep,
                              void *scratch, hipStream_t s) {
    LgArgs g = {};
    g.codes = w.codes;
    g.sc = w.scales;
    g.dst = dst;
    g.q = (const int8_t *)scratch;
    g.s = (const float *)((const uint8_t *)scratch + lg_q_bytes(w, m));
    g.m = (uint32_t)m;
    g.n = (uint32_t)w.n;
    g.n_pad = (uint32_t)w.n_pad;
    g.nsteps = lg_steps(w);
    g.nbk = (uint32_t)((w.k + w.block - 1) / w.block);
    g.mt16 = (uint32_t)((m + 15) / 16);
    g.codebook = w.codebook;
    const EpPick pk = pick_ep(ep);
    g.col_a = pk.a;
    g.col_b = pk.b;
    g.act = pk.act;
    g.act_alpha = pk.alpha;
    const int epv = pk.v == 3 ? 2 : pk.v;
    const dim3 qgrid((g.mt16 * g.nbk + 3) / 4);
    const uint32_t nslab = g.nsteps * 4;
    int8_t *q = (int8_t *)scratch;
    float *sp = (float *)((uint8_t *)scratch + lg_q_bytes(w, m));
    const bool vec = (w.k & 7) == 0 && ((uintptr_t)lhs & 15) == 0;
#define SMG_LG(SPB)                                                                                            \
    if (vec)                                                                                                   \
        hipLaunchKernelGGL((lowbit_quant_frag<SPB, true>), qgrid, dim3(256), 0, s, lhs, g.m, (uint32_t)w.k,    \
                           nslab, g.mt16, g.nbk, q, sp);                                                       \
    else                                                                                                       \
        hipLaunchKernelGGL((lowbit_quant_frag<SPB, false>), qgrid, dim3(256), 0, s, lhs, g.m, (uint32_t)w.k,   \
                           nslab, g.mt16, g.nbk, q, sp);                                                       \
    {                                                                                                          \
        const hipError_t e = hipGetLastError();                                                                \
        if (e != hipSuccess) return e;                                                                         \
    }                                                                                                          \
    return w.kind == W_Q2 ? launch_lg_rows<2, SPB>(g, ep, epv, s) : launch_lg_rows<1, SPB>(g, ep, epv, s);
    if (w.block == 64) { SMG_LG(1) }
    if (w.block == 128) { SMG_LG(2) }
    SMG_LG(4)
#undef SMG_LG
}

}  // namespace smg
