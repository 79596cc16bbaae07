// Dense f16 / bf16 GEMM with both operands' K contiguous:
// C = ep(to16(beta * A @ B)), or alpha * C + beta * A @ B, over A [m][lda] and
// B [n][ldb] (column j's K at row j): Packed<f16> / Packed<bf16>
// (Gemm::new(&a, &packed, m)...run(), replacing run_packed,
// csrc/gemm_half.h:1054) and the strided gemm_f16 / gemm_bf16
// (src/kernels/f16.rs:126-204, bf16.rs:140-200). K from 64 in multiples of 8 with
// 16-byte-aligned rows; an A of any other kind is packed into such rows first
// where that pays and there is scratch for it (dense_pack_a_bytes), else the call
// goes to gemm_kernel (gemm_mfma.hip).
// Products are v_mfma_f32_16x16x32_{f16,bf16} accumulating in f32, the portable
// path's accumulator type (src/reference.rs:349-387).
//
// gemm_dense_big: 256 x 256 tile, eight waves, two per SIMD, a 128 x 64 piece
// each. Tiles go global -> LDS by DMA (16-byte chunks swizzled: chunk c of row
// r at slot c ^ (r & 7), so fragment reads are conflict-free), two stages of 64
// depths. A step is four phases, one quarter of the wave's piece each (half of
// its rows x half of its columns, 16 products of 16x16x32 a phase):
//   phase 0 reads row half 0 and multiplies it by column half 0 (read in the
//   phase before), 1 reads column half 1, 2 row half 1, 3 the next step's
//   column half 0.
// A phase is a memory slot (its fragment reads, and two of a step's eight DMA
// instructions) and a product slot, each ended by a workgroup barrier; waves
// 4-7 run one slot behind waves 0-3, so on every SIMD one wave multiplies
// while the other reads. Each quarter of a stage is refilled as soon as both
// groups have read it, six phases (a step and a half, over 3000 cycles) before
// its next reading, and a phase waits only for the quarter the next phase
// reads: the DMA is never drained inside the loop. (128 x 256, a wave 64 x 64,
// where 256-row tiles leave compute units idle.)
// gemm_dense_tile: smaller tiles of four waves for smaller products.
// What bounds them: 8192^3 runs at 1.42 PF/s, 1.5 us a step of 64 depths where
// the products alone are 0.85 us at the nominal clock. Counters at 4096^3: the
// matrix cores busy 60 % of the kernel's cycles, waves waiting for an issue slot
// 42 % of theirs and for data or a barrier 28 %. The smaller tiles wait: 64 x 128 at
// 1000 x 3000 x 2000, the matrix cores busy 15 %, waves waiting for the next stage
// 56 %.
#include <algorithm>
#include <type_traits>

#include "dense_tile.cuh"

namespace smg {

namespace {

constexpr int DB = 256, DB_NT = 512;  // tile columns, threads
constexpr int DB_CS = DB + 8;         // halfs per staged output row
template <int BM>
struct DBig {
    static constexpr int RT = BM / 64;             // row tiles of a wave's row half
    static constexpr int AH = BM / 2 * 128;        // bytes of a row half of the tile, 64 depths
    static constexpr int BH = DB / 2 * 128;        // bytes of a column half
    static constexpr int STAGE = 2 * (AH + BH);    // row halves 0, 1, column halves 0, 1
    static constexpr int QA = RT / 2, QB = 2;      // DMA instructions a wave for a half
    static constexpr int STG = BM / 2 * DB_CS * 2; // a staged half of the output tile
    static_assert(STG + EP_FUSED * (BM + DB) * 4 <= 2 * STAGE, "the store exceeds the ring");
};

template <int BM, bool BF16, int EPV>
__global__ void __launch_bounds__(DB_NT) gemm_dense_big(DArgs g, EpArgs ep) {
    using T = DBig<BM>;
    constexpr int RT = T::RT, RH = 16 * RT;  // rows of a wave's row half
    __shared__ __align__(1024) uint8_t ring[2 * T::STAGE];
    const int t = threadIdx.x, lane = t % 64, lr = lane % 16, lg = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int wr = wave / 4, wc = wave % 4;
    uint32_t tm, tn;
    dense_tile<8>(blockIdx.x, gridDim.x, (g.m + BM - 1) / BM, (g.n + DB - 1) / DB, tm, tn);
    const uint32_t row0 = tm * BM, col0 = tn * DB;
    const uint32_t lds0 = lds_addr(ring);
    const uint32_t ksteps = (g.k + 63) / 64, last = ksteps - 1;

    // DMA sources: instruction q of a half moves its chunks (8q + wave) * 64 +
    // lane: row p / 8 of the half, slot p % 8. Half h of the rows holds rows RH h
    // .. RH h + RH - 1 of each wave row's 2 RH, half h of the columns 32h .. 32h +
    // 31 of each wave column's 64. An address is a scalar part (the
    // instruction's rows and the step) and the lane's row and chunk.
    const rsrc4_t ra = dense_rsrc(g.a, row0, g.m, g.lda, g.k), rb = dense_rsrc(g.b, col0, g.brows, g.ldb, g.k);
    const uint32_t lda2 = (uint32_t)g.lda * 2, ldb2 = (uint32_t)g.ldb * 2;
    const uint32_t chunk = (lane % 8) ^ (lane / 8);  // row % 8 is lane / 8 in every piece
    const uint32_t va = (lane / 8) * lda2 + chunk * 16, vb = (lane / 8) * ldb2 + chunk * 16;
    // half h of the rows (columns) of a step into its stage
    auto dma = [&](uint32_t step, int h, auto cols_c) __attribute__((always_inline)) {
        constexpr bool COLS = decltype(cols_c)::value;
        constexpr int Q = COLS ? T::QB : T::QA, WR = COLS ? 32 : RH;
        const uint32_t ks = min(step, last);
        const uint32_t dst = lds0 + (step & 1) * T::STAGE + (COLS ? 2 * T::AH + h * T::BH : h * T::AH) + wave * 1024;
        uint32_t v = COLS ? vb : va;
        if (ks * 64 + 64 > g.k) v = ks * 64 + chunk * 8 < g.k ? v : OOB;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const uint32_t r = (q * 8 + wave) * 8, row = (r / WR) * (2 * WR) + h * WR + r % WR;
            dma16_buf(COLS ? rb : ra, v + row * (COLS ? ldb2 : lda2) + ks * 128, dst + q * 8192);
        }
    };
    constexpr std::integral_constant<bool, false> rows;
    constexpr std::integral_constant<bool, true> cols;
    // fragment of row (column) tile i of a half, depths 32 kk ..: this lane's 16
    // bytes of row lr. (The addresses are opaque, so that the tiles are constant
    // offsets of one register instead of a register each.)
    const uint32_t f0 = lr * 128 + ((lg ^ (lr & 7)) << 4);
    const uint32_t fa = lds0 + wr * RH * 128 + f0, fb = lds0 + 2 * T::AH + wc * 32 * 128 + f0;
    auto read_a = [&](uint32_t step, int h, u32x4_t (&x)[RT][2]) __attribute__((always_inline)) {
        uint32_t b0 = fa + (step & 1) * T::STAGE + h * T::AH, b1 = b0 ^ 64;
        asm volatile("" : "+v"(b0), "+v"(b1));
#pragma unroll
        for (int i = 0; i < RT; i++) {
            x[i][0] = lds_load<u32x4_t>(b0 + i * 2048);
            x[i][1] = lds_load<u32x4_t>(b1 + i * 2048);
        }
    };
    auto read_b = [&](uint32_t step, int h, u32x4_t (&x)[2][2]) __attribute__((always_inline)) {
        uint32_t b0 = fb + (step & 1) * T::STAGE + h * T::BH, b1 = b0 ^ 64;
        asm volatile("" : "+v"(b0), "+v"(b1));
#pragma unroll
        for (int j = 0; j < 2; j++) {
            x[j][0] = lds_load<u32x4_t>(b0 + j * 2048);
            x[j][1] = lds_load<u32x4_t>(b1 + j * 2048);
        }
    };

    float4_t acc[2][2][RT][2];  // [row half][column half][row tile][column tile]
#pragma unroll
    for (int i = 0; i < 8 * RT; i++)
        acc[i / (4 * RT)][(i / (2 * RT)) % 2][(i / 2) % RT][i % 2] = (float4_t){0.f, 0.f, 0.f, 0.f};
    u32x4_t fra[RT][2], frb0[2][2][2], frb1[2][2];

    // lane: 4 consecutive columns (4 lg ..) of row lr: the columns are the
    // first operand
    auto mul = [&](float4_t (&c)[RT][2], const u32x4_t (&x)[RT][2], const u32x4_t (&y)[2][2])
        __attribute__((always_inline)) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) c[i][j] = mfma16<BF16>(y[j][kk], x[i][kk], c[i][j]);
        __builtin_amdgcn_s_setprio(0);
    };
    // the memory slot's end: this phase's reads are issued, the half that the
    // next phase reads has landed (five halves are younger)
    // (of them, the phase's own kind counts twice)
    auto mem_end = [&](auto cols_c) __attribute__((always_inline)) {
        wait_vm<2 * (T::QA + T::QB) + (decltype(cols_c)::value ? T::QB : T::QA)>();
        barrier_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    // the product slot's end: this wave's reads have completed, so the other
    // group may refill what they read
    auto mul_end = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        barrier_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](uint32_t ks, u32x4_t (&b0)[2][2], u32x4_t (&b0n)[2][2]) __attribute__((always_inline)) {
        read_a(ks, 0, fra);
        dma(ks + 1, 1, rows);
        mem_end(rows);
        mul(acc[0][0], fra, b0);
        mul_end();
        read_b(ks, 1, frb1);
        dma(ks + 2, 0, cols);
        mem_end(cols);
        mul(acc[0][1], fra, frb1);
        mul_end();
        read_a(ks, 1, fra);
        dma(ks + 2, 0, rows);
        mem_end(rows);
        mul(acc[1][1], fra, frb1);
        mul_end();
        read_b(ks + 1, 0, b0n);
        dma(ks + 2, 1, cols);
        mem_end(cols);
        mul(acc[1][0], fra, b0);
        mul_end();
    };

    dma(0, 0, cols);
    dma(0, 0, rows);
    dma(0, 1, cols);
    dma(0, 1, rows);
    dma(1, 0, cols);
    dma(1, 0, rows);
    dma(1, 1, cols);
    wait_vm<2 * (T::QA + T::QB) + T::QB>();  // step 0's first halves landed
    barrier_lds();
    read_b(0, 0, frb0[0]);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    if (wr == 1) barrier_lds();  // waves 4-7 run one slot behind
    uint32_t ks = 0;
    for (; ks + 2 <= ksteps; ks += 2) {
        step(ks, frb0[0], frb0[1]);
        step(ks + 1, frb0[1], frb0[0]);
    }
    if (ks < ksteps) step(ks, frb0[0], frb0[1]);
    if (wr == 0) barrier_lds();
    wait_vm<0>();  // the steps issued past the last
    __syncthreads();

    // (the thread's place, opaque: the loop then keeps none of what derives from
    // it for the store)
    int to = t;
    asm volatile("" : "+v"(to));
    const int lro = to % 16, lgo = to % 64 / 16;
    // Store, a row half of every wave at a time: the first RH staged
    // rows from wave row 0, the rest from wave row 1.
    uint16_t *stg = (uint16_t *)ring;
    float *colv = (float *)(ring + T::STG), *rowv = colv + EP_FUSED * DB;
    const int cl = (to % 32) * 8, rl = to / 32;
    EpCols cv;
    if constexpr (EPV == 0) ep_load_vectors<BF16, BM, DB, DB_NT>(g.st, ep, colv, rowv, row0, col0);
    if constexpr (EPV >= 2) ep_cols_load<EPV>(g.col_a, g.col_b, col0 + cl, g.n, cv);
    auto store_half = [&](const float4_t (&c)[2][RT][2], int h) __attribute__((always_inline)) {
        if (g.rd) {
#pragma unroll
            for (int w = 0; w < 2; w++)
                dense_load_c<BF16, RT>(g, stg + w * RH * DB_CS, DB_CS, rl, 16, cl, row0 + w * 2 * RH + h * RH, col0);
            __syncthreads();
        }
#pragma unroll
        for (int ch = 0; ch < 2; ch++)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    dense_stage4<BF16>(g, c[ch][i][j],
                                       stg + (wr * RH + i * 16 + lro) * DB_CS + wc * 64 + ch * 32 + j * 16 + 4 * lgo);
        __syncthreads();
#pragma unroll 1
        for (int w = 0; w < 2; w++)
            dense_store<BF16, EPV, BM, DB, RT>(g, ep, cv, colv, rowv + w * 2 * RH + h * RH, stg + w * RH * DB_CS, DB_CS, rl,
                                               16, cl, row0 + w * 2 * RH + h * RH, col0);
    };
    // (two calls, not a loop: a loop left rolled would index the accumulators
    // at run time, and keep them in memory)
    store_half(acc[0], 0);
    __syncthreads();
    store_half(acc[1], 1);
}

// The smaller tiles: BM x BN, four waves in 2 x 2, a ring of NSTG stages of 64
// depths, the DMA of step k + NSTG - 1 issued once every wave has read step k
// - 1's stage. A wave reads the next step's fragments from LDS while it
// multiplies this one's, so the ring holds one step more than the loads need.
template <int BM, int BN, int NSTG>
struct DTile {
    static constexpr int A = BM * 128, STAGE = (BM + BN) * 128, CS = BN + 8;
    static constexpr int PS = (BM + BN) / 32;  // DMA instructions a wave
    static constexpr int STORE = BM * CS * 2;
    static constexpr int LDS(int epv) {
        const int st = STORE + (epv == 0 ? EP_FUSED * (BM + BN) * 4 : 0);
        return st > NSTG * STAGE ? st : NSTG * STAGE;
    }
};

template <int BM, int BN, int NSTG, bool BF16, int EPV>
__global__ void __launch_bounds__(256, 2) gemm_dense_tile(DArgs g, EpArgs ep) {
    using T = DTile<BM, BN, NSTG>;
    constexpr int MI = BM / 32, NJ = BN / 32;  // 16 x 16 tiles of a wave's piece
    __shared__ __align__(1024) uint8_t ring[T::LDS(EPV)];
    const int t = threadIdx.x, lane = t % 64, lr = lane % 16, lg = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int wr = wave / 2, wc = wave % 2;
    uint32_t tm, tn;
    dense_tile<8>(blockIdx.x, gridDim.x, (g.m + BM - 1) / BM, (g.n + BN - 1) / BN, tm, tn);
    const uint32_t row0 = tm * BM, col0 = tn * BN;
    const uint32_t lds0 = lds_addr(ring);
    const uint32_t ksteps = (g.k + 63) / 64, last = ksteps - 1;

    const rsrc4_t ra = dense_rsrc(g.a, row0, g.m, g.lda, g.k), rb = dense_rsrc(g.b, col0, g.brows, g.ldb, g.k);
    const uint32_t lda2 = (uint32_t)g.lda * 2, ldb2 = (uint32_t)g.ldb * 2;
    const uint32_t chunk = (lane % 8) ^ (lane / 8);  // slot lane % 8 of row lane / 8 (mod 8)
    const uint32_t va = (lane / 8) * lda2 + chunk * 16, vb = (lane / 8) * ldb2 + chunk * 16;
    auto dma = [&](uint32_t step, uint32_t stage) __attribute__((always_inline)) {
        const uint32_t ks = min(step, last), dst = lds0 + stage * T::STAGE + wave * 1024;
        uint32_t v = va, w = vb;
        if (ks * 64 + 64 > g.k) {
            const bool in = ks * 64 + chunk * 8 < g.k;
            v = in ? v : OOB;
            w = in ? w : OOB;
        }
#pragma unroll
        for (int q = 0; q < MI; q++) dma16_buf(ra, v + (q * 4 + wave) * 8 * lda2 + ks * 128, dst + q * 4096);
#pragma unroll
        for (int q = 0; q < NJ; q++) dma16_buf(rb, w + (q * 4 + wave) * 8 * ldb2 + ks * 128, dst + T::A + q * 4096);
    };
    const uint32_t f0 = lr * 128 + ((lg ^ (lr & 7)) << 4);
    const uint32_t fa = lds0 + wr * (BM / 2) * 128 + f0, fb = lds0 + T::A + wc * (BN / 2) * 128 + f0;
    struct Frags {
        u32x4_t a[MI], b[NJ];
    };
    auto read = [&](uint32_t stage, int kk, Frags &f) __attribute__((always_inline)) {
        const uint32_t sb = stage * T::STAGE;
        uint32_t ba = sb + (fa ^ (kk * 64)), bb = sb + (fb ^ (kk * 64));
        asm volatile("" : "+v"(ba), "+v"(bb));  // constant offsets from here
#pragma unroll
        for (int i = 0; i < MI; i++) f.a[i] = lds_load<u32x4_t>(ba + i * 2048);
#pragma unroll
        for (int j = 0; j < NJ; j++) f.b[j] = lds_load<u32x4_t>(bb + j * 2048);
    };
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
    auto mul = [&](const Frags &f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = mfma16<BF16>(f.b[j], f.a[i], acc[i][j]);
    };

#pragma unroll
    for (int j = 0; j < NSTG - 1; j++) dma(j, j);
    wait_vm<(NSTG - 2) * T::PS>();  // step 0 landed
    barrier_lds();
    Frags h0, h1;
    read(0, 0, h0);
    uint32_t stage = 0;
    for (uint32_t ks = 0; ks < ksteps; ks++) {
        const uint32_t nstage = stage + 1 == NSTG ? 0 : stage + 1;
        read(stage, 1, h1);
        mul(h0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave has read step ks
        wait_vm<(NSTG - 3) * T::PS>();       // step ks + 1 landed
        barrier_lds();
        // every wave has read step ks - 1 (and step ks): its stage is refilled
        dma(ks + NSTG - 1, stage == 0 ? NSTG - 1 : stage - 1);
        read(nstage, 0, h0);
        mul(h1);
        stage = nstage;
    }
    wait_vm<0>();  // the steps issued past the last
    __syncthreads();

    uint16_t *stg = (uint16_t *)ring;
    float *colv = (float *)(ring + T::STORE), *rowv = colv + EP_FUSED * BN;
    constexpr int CG = BN / 8, RS = 256 / CG, R = BM / RS;
    const int cl = (t % CG) * 8, rl = t / CG;
    EpCols cv;
    if constexpr (EPV == 0) ep_load_vectors<BF16, BM, BN, 256>(g.st, ep, colv, rowv, row0, col0);
    if constexpr (EPV >= 2) ep_cols_load<EPV>(g.col_a, g.col_b, col0 + cl, g.n, cv);
    if (g.rd) {
        dense_load_c<BF16, R>(g, stg, T::CS, rl, RS, cl, row0, col0);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
            dense_stage4<BF16>(g, acc[i][j], stg + (wr * (BM / 2) + i * 16 + lr) * T::CS + wc * (BN / 2) + j * 16 + 4 * lg);
    __syncthreads();
    dense_store<BF16, EPV, BM, BN, R>(g, ep, cv, colv, rowv, stg, T::CS, rl, RS, cl, row0, col0);
}

template <int BM, bool BF16>
hipError_t launch_big(const DArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    const uint32_t tiles = ((g.m + BM - 1) / BM) * ((g.n + DB - 1) / DB);
    switch (epv) {
    case 1: hipLaunchKernelGGL((gemm_dense_big<BM, BF16, 1>), dim3(tiles), dim3(DB_NT), 0, s, g, ep); break;
    case 2: hipLaunchKernelGGL((gemm_dense_big<BM, BF16, 2>), dim3(tiles), dim3(DB_NT), 0, s, g, ep); break;
    case 3: hipLaunchKernelGGL((gemm_dense_big<BM, BF16, 3>), dim3(tiles), dim3(DB_NT), 0, s, g, ep); break;
    default: hipLaunchKernelGGL((gemm_dense_big<BM, BF16, 0>), dim3(tiles), dim3(DB_NT), 0, s, g, ep); break;
    }
    return hipGetLastError();
}
template <int BM, int BN, int NSTG, bool BF16>
hipError_t launch_tile(const DArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    const uint32_t tiles = ((g.m + BM - 1) / BM) * ((g.n + BN - 1) / BN);
    switch (epv) {
    case 1: hipLaunchKernelGGL((gemm_dense_tile<BM, BN, NSTG, BF16, 1>), dim3(tiles), dim3(256), 0, s, g, ep); break;
    case 2: hipLaunchKernelGGL((gemm_dense_tile<BM, BN, NSTG, BF16, 2>), dim3(tiles), dim3(256), 0, s, g, ep); break;
    case 3: hipLaunchKernelGGL((gemm_dense_tile<BM, BN, NSTG, BF16, 3>), dim3(tiles), dim3(256), 0, s, g, ep); break;
    default: hipLaunchKernelGGL((gemm_dense_tile<BM, BN, NSTG, BF16, 0>), dim3(tiles), dim3(256), 0, s, g, ep); break;
    }
    return hipGetLastError();
}
// The tile for an m x n x k product: the least of a cost in us, steps of 64
// depths x (full rounds of the device's compute units x occupancy, each at
// `full`; a last round of one workgroup a compute unit or fewer at `one`) +
// `fixed`, with the constants measured on 256 compute units. Measured (us, f16,
// tiles 256x256 / 128x256 / 64x128 / 64x64 / 32x64): 4096^3 105 / 145 / 181 /
// 218 / 282; 512 x 14336 x 4096 86 / 64 / 84 / 95 / 139; 2048^3 45 / 34 / 25 / 30
// / 40; 1000 x 3000 x 2000 45 / 34 / 24 / 29 / 34; 256 x 4096 x 4096 74 / 58 / 36
// / 20 / 21; 64 x 512 x 512 15 / - / 6.6 / 5.2 / 4.3. (gemm_kernel, which served
// these calls before: 197, 95, 47, 60, 80, 12.)
struct DCost {
    uint32_t bm, bn, occ;
    float one, full, fixed;
};
constexpr DCost DENSE_TILES[] = {{256, 256, 1, 1.50f, 1.50f, 8.0f},
                                 {128, 256, 1, 0.97f, 0.97f, 6.0f},
                                 {64, 128, 2, 0.53f, 0.70f, 3.0f},
                                 {64, 64, 2, 0.29f, 0.45f, 2.5f},
                                 {32, 64, 3, 0.235f, 0.43f, 2.5f}};
int dense_pick(size_t m, size_t n, size_t k) {
    const size_t cus = (size_t)device_cus(), steps = (k + 63) / 64;
    int best = 0;
    float least = 0.0f;
    for (int i = 0; i < 5; i++) {
        const DCost &c = DENSE_TILES[i];
        const size_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
        const size_t rounds = tiles / (cus * c.occ), rest = tiles % (cus * c.occ);
        const float t = (float)steps * ((float)rounds * c.full + (rest == 0 ? 0.0f : rest <= cus ? c.one : c.full)) +
                        c.fixed;
        if (i == 0 || t < least) {
            best = i;
            least = t;
        }
    }
    return best;
}
template <bool BF16>
hipError_t launch_dense_shape(const DArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    switch (dense_pick(g.m, g.n, g.k)) {
    case 0: return launch_big<256, BF16>(g, ep, epv, s);
    case 1: return launch_big<128, BF16>(g, ep, epv, s);
    case 2: return launch_tile<64, 128, 3, BF16>(g, ep, epv, s);
    case 3: return launch_tile<64, 64, 4, BF16>(g, ep, epv, s);
    default: return launch_tile<32, 64, 4, BF16>(g, ep, epv, s);
    }
}

}  // namespace

TileDims gemm_dense_tile_dims(size_t m, size_t n, size_t k) {
    const DCost &c = DENSE_TILES[dense_pick(m, n, k)];
    return {c.bm, c.bn};
}

bool gemm_dense_supported(const DenseGemm &d) {
    const size_t big = (size_t)1 << 31;
    return d.m > 0 && d.n > 0 && d.k >= 64 && d.k % 8 == 0 && d.lda % 8 == 0 && d.ldb % 8 == 0 &&
           d.lda >= (long)d.k && d.ldb >= (long)d.k && ((uintptr_t)d.a & 15) == 0 && ((uintptr_t)d.b & 15) == 0 &&
           // a tile's rows and a row's K within 2^31 bytes (past a resource's end
           // OOB plus that offset still lies past it); A as gemm_kernel takes it
           ((d.m - 1) * (size_t)d.lda + d.k) * 2 < big && (size_t)(DB + 1) * d.lda * 2 < big &&
           (size_t)(DB + 1) * d.ldb * 2 < big && d.m < big && d.n < big && d.k < big;
}

hipError_t launch_gemm_dense(const DenseGemm &d, const EpArgs &ep, bool bf16, hipStream_t s) {
    DArgs g = {};
    g.a = d.a;
    g.b = d.b;
    const bool graph = ep.n_nodes != 0;
    g.st = {d.dst, d.dst_rs, d.dst_cs, (uint32_t)d.m, (uint32_t)d.n, d.alpha, d.read_dst && graph ? 1u : 0u};
    g.beta = d.beta;
    g.alpha = d.alpha;
    g.rd = d.read_dst && !graph ? 1u : 0u;
    g.m = (uint32_t)d.m;
    g.n = (uint32_t)d.n;
    g.k = (uint32_t)d.k;
    g.brows = (uint32_t)d.brows;
    g.lda = d.lda;
    g.ldb = d.ldb;
    const EpPick pk = pick_ep(ep);
    g.col_a = pk.a;
    g.col_b = pk.b;
    g.act = pk.act;
    g.act_alpha = pk.alpha;
    const int epv = g.st.add_dst ? 0 : pk.v;
    return bf16 ? launch_dense_shape<true>(g, ep, epv, s) : launch_dense_shape<false>(g, ep, epv, s);
}

}  // namespace smg
