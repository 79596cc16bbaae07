// f16 GEMM over 2-bit / 1-bit weights: matmul_q2_mopa / matmul_q1_mopa (+ _ep)
// (src/kernels/lowbit/matmul.rs:100-139,178-197), replacing unpack_q{1,2}_f16 +
// lowbit_panels (csrc/gemm_f16f16_lowbit.h:27-194) for row-major 16-byte-aligned
// A, K in multiples of 8 and blocks of 64 or more; other calls go to
// gemm_kernel (gemm_mfma.hip). Weights are f16(scale * value), rounded once, f32
// accumulation, as there.
//
// gemm_dense_big's tile and phases (gemm_dense.cuh: BM x 256, eight waves, two
// groups one slot apart, four phases a 64-depth step), with the weights kept
// packed: a step's codes (one dword a column and 16 depths) and scales go
// global -> LDS by DMA in a ring of three, 4.5 KB a step where f16 weights are
// 32, and each wave expands the 64 columns it multiplies in registers, in the
// memory slots, beside the other group's products. 1-bit: the depths' bits moved
// to the sign places of -scale pairs, nine vector instructions for 8 weights.
// 2-bit: scale times codebook is four f16 values, kept as their low and high
// bytes; v_perm_b32 looks both up and interleaves them, twelve for 8. A column
// half's dwords are read from LDS a phase before they are expanded. Each
// quarter of A's stage is refilled as in gemm_dense_big, a step's codes six
// phases ahead.
// What bounds it: the slots that expand, which take longer than the products
// beside them (128 rows: eight 16x16x32 products a slot; 3.5 vector instructions a
// product, the matrix cores busy 29 % of the kernel's cycles). 4096 depths,
// gemm_kernel -> this (us): 1-bit 512 x 14336 82 -> 70 (with bias and silu 87 ->
// 74), 1024 x 14336 160 -> 97, 4096 x 4096 178 -> 105; 2-bit 1024 x 14336 147 ->
// 104, 4096 x 4096 160 -> 116.
// (A table of pairs looked up by one v_perm_b32, seventeen instructions for 8,
// took 1-bit 512 x 14336 from 91 to 88 where this took it to 76.)
#include <type_traits>

#include "dense_tile.cuh"

namespace smg {

namespace {

constexpr int MP = 256, MP_NT = 512;  // tile columns, threads
constexpr int MP_CS = MP + 8;         // halfs per staged output row
constexpr int MP_CODES = MP * 16, MP_W = MP_CODES + MP * 2;  // bytes of a step's codes, codes and scales

struct MopaArgs {
    DArgs d;  // b unused
    const uint8_t *codes;
    const uint16_t *sc;
    uint32_t n_pad, block_shift, codebook;
};

template <int BM>
struct MpTile {
    static constexpr int RT = BM / 64;              // row tiles of a wave's row half
    static constexpr int AH = BM / 2 * 128;         // bytes of a row half of the tile, 64 depths
    static constexpr int QA = RT / 2, QW = 3;       // DMA instructions a wave: a row half, codes and scales
    static constexpr int W0 = 4 * AH;               // two stages of A, then three of codes
    static constexpr int RING = W0 + 3 * MP_W;
    static constexpr int STG = BM / 2 * MP_CS * 2;  // a staged half of the output tile
    static constexpr int LDS(int epv) {
        const int st = STG + (epv == 0 ? EP_FUSED * (BM + MP) * 4 : 0);
        return st > RING ? st : RING;
    }
};

// KIND 2: Q2, 1: Q1.
template <int BM, int KIND, int EPV>
__global__ void __launch_bounds__(MP_NT) gemm_mopa(MopaArgs ma, EpArgs ep) {
    using T = MpTile<BM>;
    constexpr int RT = T::RT, RH = 16 * RT;  // rows of a wave's row half
    const DArgs &g = ma.d;
    __shared__ __align__(1024) uint8_t ring[T::LDS(EPV)];
    const int t = threadIdx.x, lane = t % 64, lr = lane % 16, lg = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int wr = wave / 4, wc = wave % 4;
    uint32_t tm, tn;
    dense_tile<8>(blockIdx.x, gridDim.x, (g.m + BM - 1) / BM, (g.n + MP - 1) / MP, tm, tn);
    const uint32_t row0 = tm * BM, col0 = tn * MP;
    const uint32_t lds0 = lds_addr(ring);
    const uint32_t ksteps = (g.k + 63) / 64, last = ksteps - 1;

    // A: as gemm_dense_big
    const rsrc4_t ra = dense_rsrc(g.a, row0, g.m, g.lda, g.k);
    const uint32_t lda2 = (uint32_t)g.lda * 2;
    const uint32_t chunk = (lane % 8) ^ (lane / 8);
    const uint32_t va = (lane / 8) * lda2 + chunk * 16;
    auto dma_a = [&](uint32_t step, int h) __attribute__((always_inline)) {
        const uint32_t ks = min(step, last), dst = lds0 + (step & 1) * 2 * T::AH + h * T::AH + wave * 1024;
        uint32_t v = va;
        if (ks * 64 + 64 > g.k) v = ks * 64 + chunk * 8 < g.k ? v : OOB;
#pragma unroll
        for (int q = 0; q < T::QA; q++) {
            const uint32_t r = (q * 8 + wave) * 8, row = (r / RH) * (2 * RH) + h * RH + r % RH;
            dma16_buf(ra, v + row * lda2 + ks * 128, dst + q * 8192);
        }
    };
    // Codes: instruction i of wave w moves column tile 2w + i, lane l its column
    // l / 4's quarter l % 4 of the step's slab; scales: wave w (mod 2) 128
    // columns, a pair a lane. Columns past the weights' repeat the last ones.
    uint32_t wo[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t c = min(col0 + (2 * wave + i) * 16, ma.n_pad - 16);
        wo[i] = (uint32_t)(cell_col_part(c, 0, ma.n_pad) + lane / 4) * 64 + (lane % 4) * 16;
    }
    const uint32_t so = (uint32_t)cell_col_part(min(col0 + (wave & 1) * 128 + 2 * lane, ma.n_pad - 2), 0, ma.n_pad) * 2;
    auto dma_w = [&](uint32_t step) __attribute__((always_inline)) {
        const uint32_t ks = min(step, last), dst = lds0 + T::W0 + step % 3 * MP_W;
        const uint32_t grp = KIND == 2 ? ks / 4 : ks / 8, u = KIND == 2 ? ks % 4 : ks % 8 / 2;
        const uint8_t *cp = ma.codes + cell_row_part(grp, 0, ma.n_pad) * 64 + u * 4;
#pragma unroll
        for (int i = 0; i < 2; i++) dma4(cp, wo[i], dst + (2 * wave + i) * 256);
        dma4(ma.sc + cell_row_part((ks * 64) >> ma.block_shift, 0, ma.n_pad), so, dst + MP_CODES + (wave & 1) * 256);
    };

    const uint32_t f0 = lr * 128 + ((lg ^ (lr & 7)) << 4);
    const uint32_t fa = lds0 + wr * RH * 128 + f0;
    auto read_a = [&](uint32_t step, int h, u32x4_t (&x)[RT][2]) __attribute__((always_inline)) {
        uint32_t b0 = fa + (step & 1) * 2 * T::AH + h * T::AH, b1 = b0 ^ 64;
        asm volatile("" : "+v"(b0), "+v"(b1));  // constant offsets from here
#pragma unroll
        for (int i = 0; i < RT; i++) {
            x[i][0] = lds_load<u32x4_t>(b0 + i * 2048);
            x[i][1] = lds_load<u32x4_t>(b1 + i * 2048);
        }
    };
    // column half h's dwords (16 depths of a column; this lane's 8 are its half lg
    // % 2) and scales
    struct Raw {
        uint32_t q[2][2], s[2];
    };
    const uint32_t fw = lds0 + T::W0 + (wc * 64 + lr) * 16 + (lg / 2) * 4, fs = lds0 + T::W0 + MP_CODES + (wc * 64 + lr) * 2;
    auto read_w = [&](uint32_t step, int h, Raw &r) __attribute__((always_inline)) {
        uint32_t b = fw + step % 3 * MP_W + h * 512, s = fs + step % 3 * MP_W + h * 64;
        asm volatile("" : "+v"(b), "+v"(s));
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int kk = 0; kk < 2; kk++) r.q[j][kk] = lds_load<uint32_t>(b + j * 256 + kk * 8);
            r.s[j] = lds_load<uint16_t>(s + j * 32);
        }
    };
    // the codebook as f16 pairs
    half2_t cb01, cb23;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        cb01[i] = (_Float16)(float)(int8_t)(ma.codebook >> (8 * i));
        cb23[i] = (_Float16)(float)(int8_t)(ma.codebook >> (8 * (i + 2)));
    }
    const uint32_t sub = KIND == 2 ? (lg & 1) * 4 : (lg & 1) * 2;
    auto expand = [&](uint32_t step, const Raw &r, u32x4_t (&y)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t s2 = r.s[j] | (r.s[j] << 16);
            if constexpr (KIND == 2) {
                const uint32_t t01 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, s2) * cb01);
                const uint32_t t23 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, s2) * cb23);
                const uint32_t tl = __builtin_amdgcn_perm(t23, t01, 0x06040200u);  // the four values' low bytes
                const uint32_t th = __builtin_amdgcn_perm(t23, t01, 0x07050301u);  // and high bytes
#pragma unroll
                for (int kk = 0; kk < 2; kk++)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const uint32_t c = (r.q[j][kk] >> (sub + 2 * i)) & 0x03030303u;
                        const uint32_t lo = __builtin_amdgcn_perm(tl, tl, c), hi = __builtin_amdgcn_perm(th, th, c);
                        y[j][kk][2 * i] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
                        y[j][kk][2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
                    }
            } else {
                // the depths' bits moved to the sign places of -scale pairs
                const uint32_t sn = s2 ^ 0x80008000u;
#pragma unroll
                for (int kk = 0; kk < 2; kk++) {
                    const uint32_t w = r.q[j][kk] << (6 - sub - 4 * (step & 1));
                    const uint32_t p01 = __builtin_amdgcn_perm(w, w, 0x010C000Cu);
                    const uint32_t p23 = __builtin_amdgcn_perm(w, w, 0x030C020Cu);
                    y[j][kk][0] = ((p01 << 1) & 0x80008000u) ^ sn;
                    y[j][kk][1] = ((p23 << 1) & 0x80008000u) ^ sn;
                    y[j][kk][2] = (p01 & 0x80008000u) ^ sn;
                    y[j][kk][3] = (p23 & 0x80008000u) ^ sn;
                }
            }
        }
    };

    float4_t acc[2][2][RT][2];  // [row half][column half][row tile][column tile]
#pragma unroll
    for (int i = 0; i < 8 * RT; i++)
        acc[i / (4 * RT)][(i / (2 * RT)) % 2][(i / 2) % RT][i % 2] = (float4_t){0.f, 0.f, 0.f, 0.f};
    u32x4_t fra[RT][2], frb0[2][2][2], frb1[2][2];
    Raw raw;
    auto mul = [&](float4_t (&c)[RT][2], const u32x4_t (&x)[RT][2], const u32x4_t (&y)[2][2])
        __attribute__((always_inline)) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) c[i][j] = mfma16<false>(y[j][kk], x[i][kk], c[i][j]);
        __builtin_amdgcn_s_setprio(0);
    };
    auto mem_end = [&]() __attribute__((always_inline)) {
        barrier_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    // what the next phase reads has landed: of A's halves and the codes, two
    // halves and one step's codes are younger
    auto landed = [&]() __attribute__((always_inline)) { wait_vm<2 * T::QA + T::QW>(); };
    auto mul_end = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        barrier_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](uint32_t ks, u32x4_t (&b0)[2][2], u32x4_t (&b0n)[2][2]) __attribute__((always_inline)) {
        read_a(ks, 0, fra);
        read_w(ks, 1, raw);
        dma_a(ks + 1, 1);
        mem_end();
        mul(acc[0][0], fra, b0);
        mul_end();
        expand(ks, raw, frb1);
        dma_w(ks + 2);
        landed();  // row half 1 of step ks, the codes of step ks + 1
        mem_end();
        mul(acc[0][1], fra, frb1);
        mul_end();
        read_a(ks, 1, fra);
        read_w(ks + 1, 0, raw);
        dma_a(ks + 2, 0);
        mem_end();
        mul(acc[1][1], fra, frb1);
        mul_end();
        expand(ks + 1, raw, b0n);
        landed();  // row half 0 of step ks + 1
        mem_end();
        mul(acc[1][0], fra, b0);
        mul_end();
    };

    dma_w(0);
    dma_a(0, 0);
    dma_a(0, 1);
    dma_w(1);
    dma_a(1, 0);
    landed();  // step 0's codes and row half 0
    barrier_lds();
    read_w(0, 0, raw);
    expand(0, raw, frb0[0]);
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

    // store: as gemm_dense_big
    int to = t;
    asm volatile("" : "+v"(to));
    const int lro = to % 16, lgo = to % 64 / 16;
    uint16_t *stg = (uint16_t *)ring;
    float *colv = (float *)(ring + T::STG), *rowv = colv + EP_FUSED * MP;
    const int cl = (to % 32) * 8, rl = to / 32;
    EpCols cv;
    if constexpr (EPV == 0) ep_load_vectors<false, BM, MP, MP_NT>(g.st, ep, colv, rowv, row0, col0);
    if constexpr (EPV >= 2) ep_cols_load<EPV>(g.col_a, g.col_b, col0 + cl, g.n, cv);
    auto store_half = [&](const float4_t (&c)[2][RT][2], int h) __attribute__((always_inline)) {
#pragma unroll
        for (int ch = 0; ch < 2; ch++)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    dense_stage4<false>(g, c[ch][i][j],
                                        stg + (wr * RH + i * 16 + lro) * MP_CS + wc * 64 + ch * 32 + j * 16 + 4 * lgo);
        __syncthreads();
#pragma unroll 1
        for (int w = 0; w < 2; w++)
            dense_store<false, EPV, BM, MP, RT>(g, ep, cv, colv, rowv + w * 2 * RH + h * RH, stg + w * RH * MP_CS, MP_CS,
                                                rl, 16, cl, row0 + w * 2 * RH + h * RH, col0);
    };
    store_half(acc[0], 0);
    __syncthreads();
    store_half(acc[1], 1);
}

template <int BM, int KIND>
hipError_t launch_mp(const MopaArgs &g, const EpArgs &ep, int epv, hipStream_t s) {
    const uint32_t tiles = ((g.d.m + BM - 1) / BM) * ((g.d.n + MP - 1) / MP);
    switch (epv) {
    case 1: hipLaunchKernelGGL((gemm_mopa<BM, KIND, 1>), dim3(tiles), dim3(MP_NT), 0, s, g, ep); break;
    case 2: hipLaunchKernelGGL((gemm_mopa<BM, KIND, 2>), dim3(tiles), dim3(MP_NT), 0, s, g, ep); break;
    case 3: hipLaunchKernelGGL((gemm_mopa<BM, KIND, 3>), dim3(tiles), dim3(MP_NT), 0, s, g, ep); break;
    default: hipLaunchKernelGGL((gemm_mopa<BM, KIND, 0>), dim3(tiles), dim3(MP_NT), 0, s, g, ep); break;
    }
    return hipGetLastError();
}

// The tile's rows, or 0 where gemm_kernel is faster. Rounds: a workgroup fills a
// compute unit, so a product takes as many passes over the chip as its tiles
// make. A pass over 4096 depths, us:
//   Q1: 128 rows 65 (few tiles) - 76 (all units busy), 256 rows 83 - 92,
//       gemm_kernel (256 x 128) 70 - 90 -> 128 rows, or 256 where those need
//       fewer rounds by more than 5 : 4;
//   Q2: 256 rows 99 - 105, gemm_kernel 68 - 86, 128 rows of this 83 - 87 ->
//       256 rows where gemm_kernel's rounds are more by 5 : 4. (Seventeen or
//       twelve instructions for 8 weights took Q2 the same time; both look up
//       with eight v_perm_b32, Q1 with two, so those seem to set its pace.)
// Up to 128 rows gemm_kernel's 128 x 128 tiles take as long (1-bit 4096 x 4096,
// 16 rows: 64 against 65).
int mopa_tile(const WDev &w, size_t m) {
    if (m <= 128) return 0;
    const size_t cus = (size_t)device_cus();
    const size_t nt = (w.n + MP - 1) / MP, mt = (m + 255) / 256;
    const size_t r256 = (mt * nt + cus - 1) / cus, r128 = ((m + 127) / 128 * nt + cus - 1) / cus,
                 rk = (mt * ((w.n + 127) / 128) + cus - 1) / cus;
    if (w.kind == W_Q1) return r256 * 5 < r128 * 4 ? 256 : 128;
    return r256 * 5 < rk * 4 ? 256 : 0;
}

}  // namespace

TileDims gemm_mopa_tile(const WDev &w, size_t m) {
    const uint32_t rows = (uint32_t)mopa_tile(w, m);
    return {rows, rows ? (uint32_t)MP : 0u};
}

bool gemm_mopa_supported(const WDev &w, size_t m, long lhs_cs, long lhs_rs, const uint16_t *lhs) {
    const size_t big = (size_t)1 << 31;
    return (w.kind == W_Q2 || w.kind == W_Q1) && m < big && w.n >= 1 && w.k >= 64 && w.k % 8 == 0 && w.block >= 64 &&
           lhs_cs == 1 && lhs_rs % 8 == 0 && lhs_rs >= (long)w.k && ((uintptr_t)lhs & 15) == 0 &&
           ((m - 1) * (size_t)lhs_rs + w.k) * 2 < big && (size_t)257 * lhs_rs * 2 < big && w.n_pad * 256 < big &&
           ((m + 127) / 128) * ((w.n + MP - 1) / MP) < big && mopa_tile(w, m) != 0;
}

// Whether the call's store leaves the product's gain. A tile stores 256 columns on
// one compute unit where gemm_kernel's 128-column tiles use two, so a store that
// takes long -- an interpreted graph with tensors or many nodes, an activation on
// libm's exponentials -- needs more depth or a grid that fills the device.
// gemm_kernel -> this (us), 1-bit: 129 x 128 x 512 with a tensor 22.6 -> 25.5, with
// mish 36 -> 51, but with a row product 18.6 -> 17.8; 200 x 1000 x 1024 34.4 -> 36.6,
// 54 -> 60, 29.0 -> 26.4, x 2048 50.2 -> 51.8, 70 -> 76; 300 x 4096 x 2048 52.7 ->
// 52.6, 80 -> 76; 600 x 9000 x 1024 (180 tiles) 41.9 -> 40.1, 67 -> 63. 2-bit (256-row
// tiles) 2100 x 4096 x 512 48.1 -> 53.0, 82 -> 94, 39.1 -> 28.1, x 1024 66.3 -> 65.5,
// 100 -> 108.
bool gemm_mopa_pays(const WDev &w, size_t m, const EpArgs &ep) {
    bool longer = false, exps = false;
    if (pick_ep(ep).v == 0) longer = ep.n_nodes > 4;
    for (uint32_t i = 0; i < ep.n_nodes; i++) {
        longer |= ep.cls[i] == EPC_TENSOR;
        exps |= ep.fam[i] == EPF_ACT && ep.nodes[i].aux >= EP_ACT_EXP;
    }
    if (!longer && !exps) return true;
    const size_t tiles = ((m + 127) / 128) * ((w.n + MP - 1) / MP);
    if (w.k >= 4096 || (w.k >= 2048 && tiles >= 32)) return true;
    if (tiles * 2 < (size_t)device_cus()) return false;
    return exps ? mopa_tile(w, m) == 128 : w.k >= 1024;
}

hipError_t launch_gemm_mopa(const WDev &w, size_t m, uint16_t *dst, long dst_cs, long dst_rs, const uint16_t *lhs,
                            long lhs_rs, float beta, const EpArgs &ep, hipStream_t s) {
    MopaArgs g = {};
    g.d.a = lhs;
    g.d.st = {dst, dst_rs, dst_cs, (uint32_t)m, (uint32_t)w.n, 0.0f, 0u};
    g.d.beta = beta;
    g.d.m = (uint32_t)m;
    g.d.n = (uint32_t)w.n;
    g.d.k = (uint32_t)w.k;
    g.d.lda = lhs_rs;
    const EpPick pk = pick_ep(ep);
    g.d.col_a = pk.a;
    g.d.col_b = pk.b;
    g.d.act = pk.act;
    g.d.act_alpha = pk.alpha;
    g.codes = w.codes;
    g.sc = w.scales;
    g.n_pad = (uint32_t)w.n_pad;
    g.block_shift = (uint32_t)__builtin_ctzll(w.block);
    g.codebook = w.codebook;
    if (w.kind == W_Q2) return launch_mp<256, 2>(g, ep, pk.v, s);
    return mopa_tile(w, m) == 256 ? launch_mp<256, 1>(g, ep, pk.v, s) : launch_mp<128, 1>(g, ep, pk.v, s);
}

}  // namespace smg
