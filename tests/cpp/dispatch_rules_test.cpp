// The dispatch rules' bounds on sizes whose arrays need not exist: only host
// code of the launch interface runs, nothing reaches a GPU.
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "kernels.h"

using namespace smg;

static int failed = 0;
#define CHECK(c)                                                  \
    do {                                                          \
        if (!(c)) {                                               \
            std::printf("line %d: %s does not hold\n", __LINE__, #c); \
            failed++;                                             \
        }                                                         \
    } while (0)

static WDev lowbit(int kind, size_t n, size_t k, size_t block) {
    const size_t group = kind == W_Q2 ? Q2_GROUP : Q1_GROUP;
    WDev w = {};
    w.kind = kind;
    w.n = n;
    w.k = k;
    w.block = block;
    w.n_pad = (n + 127) / 128 * 128;
    w.nchunks = (k + group - 1) / group;
    w.sc_rows = (k + block - 1) / block;
    return w;
}

// Byte offset of the last column's codes from the first's, as a GEMM lane
// adds it to its step's base.
static size_t last_code(const WDev &w) { return cell_col_part(w.n_pad - 1, 0, w.n_pad) * 64 + 3 * 16 + 16; }

// `tiles`: a call a line on stdin ("dense m n k", "lowbit bits block m n k", "mopa
// bits m n k"), its tile ("rows cols") a line on stdout.
static int tiles() {
    char op[16];
    size_t m, n, k, block;
    int bits;
    while (std::scanf("%15s", op) == 1) {
        TileDims t = {0, 0};
        if (!std::strcmp(op, "dense")) {
            if (std::scanf("%zu %zu %zu", &m, &n, &k) != 3) return 1;
            t = gemm_dense_tile_dims(m, n, k);
        } else if (!std::strcmp(op, "lowbit")) {
            if (std::scanf("%d %zu %zu %zu %zu", &bits, &block, &m, &n, &k) != 5) return 1;
            t = lowbit_gemm_tile(lowbit(bits == 1 ? W_Q1 : W_Q2, n, k, block), m);
        } else if (!std::strcmp(op, "mopa")) {
            if (std::scanf("%d %zu %zu %zu", &bits, &m, &n, &k) != 4) return 1;
            t = gemm_mopa_tile(lowbit(bits == 1 ? W_Q1 : W_Q2, n, k, 128), m);
        } else {
            return 1;
        }
        std::printf("%u %u\n", t.rows, t.cols);
    }
    return 0;
}

int main(int argc, char **argv) {
    if (argc > 1 && !std::strcmp(argv[1], "tiles")) return tiles();
    const int kinds[2] = {W_Q2, W_Q1};
    // The many-row GEMM serves a call only where a column's code offset fits the
    // DMA's 32-bit lane offset.
    for (int kind : kinds)
        for (size_t block : {(size_t)64, (size_t)128, (size_t)256})
            for (size_t n : {(size_t)1, (size_t)11008, ((size_t)1 << 23) - 128, (size_t)1 << 23, ((size_t)1 << 24) - 1,
                             (size_t)1 << 24, ((size_t)1 << 24) + 1, (size_t)1 << 25, (size_t)1 << 27}) {
                const WDev w = lowbit(kind, n, 64, block);
                const size_t bytes = lowbit_gemm_bytes(w, 9);
                CHECK(bytes == 0 || last_code(w) <= 0xFFFFFFFFu);
                CHECK(n >= ((size_t)1 << 23) || bytes != 0);  // ordinary widths stay on it
                const uint16_t *a = (const uint16_t *)256;
                CHECK(!gemm_mopa_supported(w, 512, 1, 64, a) || last_code(w) <= 0xFFFFFFFFu);
            }

    // Blocks of 256, past 2048 depths, few rows, one round of GEMV workgroups: the
    // GEMV; each limit by one step on either side.
    for (int kind : kinds) {
        const size_t calls[][4] = {{9, 700, 8000, 1},   {9, 700, 2048, 0},   {9, 700, 2049, 1},   {32, 2048, 4096, 1},
                                   {33, 2048, 4096, 0}, {16, 4096, 4096, 1}, {16, 4097, 4096, 0}, {64, 1024, 8192, 1},
                                   {65, 128, 8192, 0},  {33, 128, 8193, 0},  {32, 128, 8193, 1}};
        for (const auto &c : calls) {
            CHECK((lowbit_gemm_bytes(lowbit(kind, c[1], c[2], 256), c[0]) == 0) == (c[3] != 0));
            CHECK(lowbit_gemm_bytes(lowbit(kind, c[1], c[2], 128), c[0]) != 0);
            CHECK(lowbit_gemm_bytes(lowbit(kind, c[1], c[2], 64), c[0]) != 0);
        }
    }
    // Dense products: an A is packed where the tiles cannot read it and packing
    // pays. K < 64 alone is no reason (gemm_kernel reads such rows by vectors)
    // until gemm_kernel's own tiles need a second round.
    for (size_t k : {(size_t)1, (size_t)8, (size_t)31, (size_t)32, (size_t)56, (size_t)63, (size_t)64, (size_t)72,
                     (size_t)1001})
        for (size_t m : {(size_t)1, (size_t)16, (size_t)500, (size_t)3000})
            for (size_t n : {(size_t)100, (size_t)500, (size_t)3000}) {
                WDev w = {};
                w.kind = W_F16;
                w.n = n;
                w.k = k;
                w.n_pad = (n + 127) / 128 * 128;
                w.k_pad = (k + 63) / 64 * 64;
                w.dense = (const uint16_t *)4096;
                const uint16_t *a = (const uint16_t *)256;
                const bool vec = k % 8 == 0, two = m * n >= (size_t)9000000;
                CHECK((dense_pack_a_bytes(w, m, a, 1, (long)k) != 0) == (!vec || (k < 64 && two)));
                CHECK(dense_pack_a_bytes(w, m, a + 1, 1, (long)k) != 0);         // unaligned rows
                CHECK(dense_pack_a_bytes(w, m, a, (long)m, 1) != 0 || (m == 1 && k == 1));  // a column stride
            }
    // A strided call packs A too, but for few short rows.
    {
        const size_t calls[][4] = {{32, 300, 127, 0}, {32, 300, 129, 1}, {33, 300, 63, 0},  {33, 300, 65, 1},
                                   {200, 64, 63, 0},  {61, 499, 63, 1},  {1, 100, 8, 0},    {16, 500, 200, 1},
                                   {128, 128, 63, 0}, {129, 128, 63, 1}, {3000, 500, 3001, 1}};
        for (const auto &c : calls) {
            WDev w = {};
            w.kind = W_F16;
            w.n = c[1];
            w.k = c[2];
            w.n_pad = (c[1] + 127) / 128 * 128;
            w.k_pad = (c[2] + 63) / 64 * 64;
            w.dense = (const uint16_t *)4096;
            const uint16_t *a = (const uint16_t *)256;
            CHECK((strided_pack_a_bytes(w, c[0], a, (long)c[0], 1) != 0) == (c[3] != 0));
        }
    }
    // Low-bit f16 products: what the tile serves, a long interpreted store aside.
    {
        const auto graph = [](std::initializer_list<uint32_t> ops, uint32_t act = 0) {
            EpArgs ep = {};
            for (uint32_t op : ops) {
                ep.nodes[ep.n_nodes].op = op;
                ep.nodes[ep.n_nodes].ptr = (const void *)256;
                ep.fam[ep.n_nodes] = ep_family(op);
                ep.cls[ep.n_nodes] = ep_class(op);
                ep.n_nodes++;
            }
            if (act) {
                ep.nodes[ep.n_nodes].op = EP_OP_ACT;
                ep.nodes[ep.n_nodes].aux = act;
                ep.fam[ep.n_nodes] = ep_family(EP_OP_ACT);
                ep.cls[ep.n_nodes] = ep_class(EP_OP_ACT);
                ep.n_nodes++;
            }
            return ep;
        };
        const EpArgs none = graph({}), bias = graph({EP_OP_ADD_COL}, EP_ACT_SILU), row = graph({EP_OP_MUL_ROW}),
                     rtanh = graph({EP_OP_MUL_ROW}, EP_ACT_TANH), tensor = graph({EP_OP_ADD_COL, EP_OP_ADD_TENSOR}),
                     five = graph({EP_OP_MUL_ROW, EP_OP_ADD_ROW, EP_OP_MUL_ROW, EP_OP_ADD_ROW, EP_OP_MUL_ROW}),
                     mish = graph({EP_OP_MUL_ROW}, EP_ACT_MISH), bmish = graph({EP_OP_ADD_COL}, EP_ACT_MISH);
        const struct {
            int kind;
            size_t m, n, k;
            bool longer, exps;  // whether such graphs stay
        } calls[] = {{W_Q1, 129, 128, 512, false, false},    {W_Q1, 200, 1000, 2048, false, false},
                     {W_Q1, 200, 1000, 4096, true, true},    {W_Q1, 300, 4096, 2047, false, false},
                     {W_Q1, 300, 4096, 2048, true, true},    {W_Q1, 600, 9000, 512, false, true},
                     {W_Q1, 600, 9000, 1024, true, true},    {W_Q1, 2100, 4096, 512, false, false},
                     {W_Q2, 2100, 4096, 1024, true, false},  {W_Q2, 2100, 4096, 2048, true, true}};
        for (const auto &c : calls) {
            const WDev w = lowbit(c.kind, c.n, c.k, 128);
            for (const EpArgs *e : {&none, &bias, &row, &rtanh}) CHECK(gemm_mopa_pays(w, c.m, *e));
            for (const EpArgs *e : {&tensor, &five}) CHECK(gemm_mopa_pays(w, c.m, *e) == c.longer);
            for (const EpArgs *e : {&mish, &bmish}) CHECK(gemm_mopa_pays(w, c.m, *e) == c.exps);
        }
    }
    // Attention of row blocks: few short rows of a wide head stay on
    // attn_rows_mfma, as does what attn_rows_dma cannot address.
    {
        const struct {
            uint32_t heads, kv, hd, start, rows, staged;
        } calls[] = {{16, 8, 128, 0, 64, 0},  {16, 8, 128, 128, 64, 0}, {16, 8, 128, 129, 64, 1}, {16, 8, 128, 0, 65, 1},
                     {32, 8, 128, 160, 32, 0}, {32, 8, 128, 161, 32, 1}, {12, 12, 64, 0, 32, 1},  {12, 12, 72, 0, 32, 0},
                     {4, 4, 256, 4096, 512, 0}, {32, 8, 128, 4096, 512, 1}, {6, 1, 128, 0, 32, 0}};
        for (const auto &c : calls) {
            AttnArgs a = {};
            a.q = a.k = a.v = (const uint16_t *)256;
            a.out = (void *)512;
            a.heads = c.heads;
            a.group = c.heads / c.kv;
            a.hd = c.hd;
            a.ld = c.kv * c.hd;
            a.len = c.start + 1;
            a.rows = c.rows;
            CHECK(attn_rows_staged(a) == (c.staged != 0));
            a.out = (void *)516;
            CHECK(!attn_rows_staged(a));
        }
    }
    if (failed == 0) std::printf("dispatch rules ok\n");
    return failed != 0;
}
