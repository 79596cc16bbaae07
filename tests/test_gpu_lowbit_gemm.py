"""The many-row 2-bit / 1-bit int8 GEMM (lowbit_gemm) against the oracle, bit
for bit: quantization, block sums, the in-order fold and the op-graph are the
same steps as the decode kernels', so every output is identical."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, n, k): the fewest rows served, 16-row tile edges, 32- and 64-row tile
# edges, ragged N (one 128-column tile and several) and K below, at and past a
# 256-depth step and a Q1 group (512), K not a multiple of 8 (the element-wise
# row loads) and several steps with a last partial block
SHAPES = [(9, 128, 256), (16, 5, 64), (17, 130, 300), (31, 257, 512), (32, 384, 1024), (33, 1000, 777),
          (63, 128, 4096), (64, 129, 520), (65, 640, 2049), (130, 300, 1288),
          # 32-row, 64-row and 64 x 128 tiles (more 16-row tiles than the
          # device takes at once), ragged rows and columns
          (130, 8200, 300), (300, 8900, 256), (300, 9001, 256), (400, 16300, 328)]
# the same three tiles, one block deep (test_host_logic.py holds the rule to both)
WIDE = [(130, 8200, 128), (300, 8900, 128), (400, 16300, 128)]
BOOKS = [(-1, 0, 1, 0), (-2, -1, 1, 2), (-128, 127, 3, -7)]


def _inputs(orc, rng, m, n, k, block, bits):
    nbk = -(-k // block)
    scales = orc.f32_to_f16(rng.uniform(-0.05, 0.05, n * nbk).astype(np.float32))
    a = orc.f32_to_f16(rng.standard_normal(m * k).astype(np.float32))
    codes = rng.integers(0, 256, (k * n * bits + 7) // 8, dtype=np.uint8)
    return a, codes, scales


def _both(smg, orc, a, codes2, signs, scales, m, n, k, block, book, ep=None, nodes=(), act=None):
    q2 = smg.Q2Weights(codes2, scales, n, k, smg.Q2Params(block).with_codebook(book))
    got = np.full(m * n, 0x4880, np.uint16)
    smg.matmul_q2_ep(a, q2, got, m, ep or smg.Epilogue())
    want = orc.matmul_lowbit_ep(2, a, codes2, scales, m, n, k, block, nodes, act, codebook=book)
    assert np.array_equal(got, want), "q2"
    for layout in (smg.WeightLayout.OutIn, smg.WeightLayout.InOut):
        q1 = smg.Q1Weights(signs, scales, layout, n, k, block)
        got = np.full(m * n, 0x4880, np.uint16)
        smg.matmul_q1_ep(a, q1, got, m, ep or smg.Epilogue())
        want = orc.matmul_lowbit_ep(1, a, signs, scales, m, n, k, block, nodes, act,
                                    inout=layout == smg.WeightLayout.InOut)
        assert np.array_equal(got, want), f"q1 layout {layout}"


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("si", range(len(SHAPES)))
def test_many_rows_match_reference_bits(smg, orc, si, block):
    m, n, k = SHAPES[si]
    rng = np.random.default_rng(1000 * block + si)
    a, codes2, scales = _inputs(orc, rng, m, n, k, block, 2)
    signs = rng.integers(0, 256, (k * n + 7) // 8, dtype=np.uint8)
    _both(smg, orc, a, codes2, signs, scales, m, n, k, block, BOOKS[si % 3])


@pytest.mark.parametrize("graph", ["bias", "bias_silu", "scale_bias_gelu", "interpreted"])
def test_many_rows_epilogue_bits(smg, orc, graph):
    """Each compiled store and the interpreted one, over ragged edges."""
    m, n, k, block = 70, 203, 640, 128
    rng = np.random.default_rng(77)
    a, codes2, scales = _inputs(orc, rng, m, n, k, block, 2)
    signs = rng.integers(0, 256, (k * n + 7) // 8, dtype=np.uint8)
    b = orc.f32_to_f16(rng.uniform(-4, 4, n).astype(np.float32))
    s = orc.f32_to_f16(rng.uniform(0.5, 1.5, n).astype(np.float32))
    r = orc.f32_to_f16(rng.uniform(0.5, 1.5, m).astype(np.float32))
    t = orc.f32_to_f16(rng.uniform(-1, 1, m * n).astype(np.float32))
    ep, nodes, act = {
        "bias": (smg.Epilogue().add_col(b), [(4, 0, 0.0, b, 0)], None),
        "bias_silu": (smg.Epilogue().add_col(b).silu(), [(4, 0, 0.0, b, 0)], 3),
        "scale_bias_gelu": (smg.Epilogue().mul_col(s).add_col(b).gelu(),
                            [(5, 0, 0.0, s, 0), (4, 0, 0.0, b, 0)], 2),
        "interpreted": (smg.Epilogue().mul_row(r).add_tensor(t).sigmoid(),
                        [(3, 0, 0.0, r, 0), (6, 0, 0.0, t, n)], 5),
    }[graph]
    _both(smg, orc, a, codes2, signs, scales, m, n, k, block, (-1, 0, 1, 0), ep, nodes, act)


@pytest.mark.parametrize("graph", ["scale_bias_gelu", "interpreted"])
@pytest.mark.parametrize("m,n,k", WIDE)
def test_wide_tiles_epilogue_bits(smg, orc, m, n, k, graph):
    """The compiled and the interpreted store of the tiles past 16 rows."""
    block = 128
    rng = np.random.default_rng(m)
    a, codes, scales = _inputs(orc, rng, m, n, k, block, 2)
    b = orc.f32_to_f16(rng.uniform(-4, 4, n).astype(np.float32))
    s = orc.f32_to_f16(rng.uniform(0.5, 1.5, n).astype(np.float32))
    r = orc.f32_to_f16(rng.uniform(0.5, 1.5, m).astype(np.float32))
    if graph == "interpreted":
        ep, nodes, act = smg.Epilogue().mul_row(r).add_col(b).relu(), [(3, 0, 0.0, r, 0), (4, 0, 0.0, b, 0)], 1
    else:
        ep, nodes, act = smg.Epilogue().mul_col(s).add_col(b).gelu(), [(5, 0, 0.0, s, 0), (4, 0, 0.0, b, 0)], 2
    w = smg.Q2Weights(codes, scales, n, k, smg.Q2Params(block))
    got = np.full(m * n, 0x4880, np.uint16)
    smg.matmul_q2_ep(a, w, got, m, ep)
    assert np.array_equal(got, orc.matmul_lowbit_ep(2, a, codes, scales, m, n, k, block, nodes, act))


@pytest.mark.parametrize("m,n", [(21, 77), (130, 8200)])
def test_interpreted_store_every_node_bits(smg, orc, m, n):
    """Graphs the stores are not compiled for: every activation last and, the
    in-order ones, before another node; every operation with a scalar, row, column
    and strided tensor operand. Ragged edges, one tile and many. (Where the
    reference gives NaN, NaN.)"""
    k, block, ld = 64, 64, n + 3
    rng = np.random.default_rng(n)
    a, codes, scales = _inputs(orc, rng, m, n, k, block, 2)
    w = smg.Q2Weights(codes, scales, n, k, smg.Q2Params(block))
    half = lambda lo, hi, size: orc.f32_to_f16(rng.uniform(lo, hi, size).astype(np.float32))  # noqa: E731
    r, c, t = half(0.5, 1.5, m), half(-2, 2, n), half(0.5, 2, (m - 1) * ld + n)
    plain = np.zeros(m * n, np.uint16)
    smg.matmul_q2(a, w, plain, m)
    few = m * n > 100000  # the oracle's time
    graphs = []
    for name, kind in smg.EP_ACT.items():
        alpha = 0.3 if name in ("leaky_relu", "elu") else 0.0
        arg = (0.3,) if alpha else ()
        if few and kind not in (2, 3, 18):
            continue
        if kind <= 5:
            graphs.append((getattr(smg.Epilogue().add_scalar(0.25), name)(), [(0, 0, 0.25, None, 0)], kind))
            continue
        node = (8, kind, float(np.float32(alpha)), None, 0)
        graphs.append((getattr(smg.Epilogue().mul_row(r), name)(*arg), [(3, 0, 0.0, r, 0), node], None))
        graphs.append((getattr(smg.Epilogue(), name)(*arg).mul_row(r), [node, (3, 0, 0.0, r, 0)], None))
    for op in ("add", "sub", "mul", "div", "max", "min"):
        g, nodes = smg.Epilogue(), []
        for kind, v, s in (("scalar", None, 0.75), ("row", r, 0.0), ("col", c, 0.0), ("tensor", t, 0.0)):
            f = g.max if (op, kind) == ("max", "scalar") else g.min if (op, kind) == ("min", "scalar") else getattr(
                g, f"{op}_{kind}")
            g = f(s) if v is None else f(v, ld=ld) if kind == "tensor" else f(v)
            nodes.append((smg.EP_OP[f"{op}_{kind}"], 0, s, v, ld if kind == "tensor" else 0))
        graphs.append((g, nodes, None))
    nan = lambda x: (x & 0x7FFF) > 0x7C00  # noqa: E731
    for ep, nodes, act in graphs:
        got = np.full(m * n, 0x4880, np.uint16)
        smg.matmul_q2_ep(a, w, got, m, ep)
        want = orc.apply_ep(plain, m, n, nodes, act)
        assert np.array_equal(nan(got), nan(want)), nodes
        assert np.array_equal(got[~nan(want)], want[~nan(want)]), (nodes, act)


def test_many_rows_special_activations(smg, orc):
    """Blocks of zeros, infinities, NaN and the smallest subnormals, and rows
    that differ only in one block: amax, inv and s as quantize_row gives them
    (NaN outputs compared as NaN: their bits are the platform's)."""
    m, n, k, block = 40, 130, 512, 128
    rng = np.random.default_rng(5)
    a, codes2, scales = _inputs(orc, rng, m, n, k, block, 2)
    av = a.reshape(m, k)
    av[1, :128] = 0
    av[2, 130] = 0x7C00
    av[3, 260] = 0x7E00
    av[4, 384:] = 1
    av[5, :] = 0x7BFF
    av[17, 0] = 0xFC00
    av[33, 511] = 0xFE01
    q2 = smg.Q2Weights(codes2, scales, n, k, smg.Q2Params(block))
    got = np.zeros(m * n, np.uint16)
    smg.matmul_q2(a, q2, got, m)
    want = orc.lowbit_reference(2, a, codes2, scales, m, n, k, block)
    nan = lambda x: (x & 0x7FFF) > 0x7C00  # noqa: E731
    assert np.array_equal(nan(got), nan(want))
    assert np.array_equal(got[~nan(want)], want[~nan(want)])


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("m,n,k", [(70, 200, 512), (21, 130, 1001), (16, 64, 65)])
def test_many_rows_of_an_unaligned_a(smg, orc, m, n, k, block):
    """An A off 16-byte alignment, NaN around it: the rows' staged form, the same
    bits as the oracle's."""
    import torch
    rng = np.random.default_rng(k + block)
    a, codes, scales = _inputs(orc, rng, m, n, k, block, 2)
    w = smg.Q2Weights(codes, scales, n, k, smg.Q2Params(block))
    buf = torch.full((m * k + 16,), 0x7E00, dtype=torch.int16, device="cuda")
    ad = buf[3:3 + m * k]
    ad.copy_(torch.from_numpy(a.view(np.int16)))
    c = torch.zeros(m * n, dtype=torch.int16, device="cuda")
    smg.matmul_q2(ad, w, c, m)
    want = orc.lowbit_reference(2, a, codes, scales, m, n, k, block)
    assert np.array_equal(c.cpu().numpy().view(np.uint16), want)


def test_noalloc_keeps_the_calls_it_took(smg, orc):
    """961 rows at K = 4096: the GEMM's scratch (16-row tiles) would pass the
    static array, the GEMV's fits it -- the call runs there, the same bits."""
    import torch
    m, n, k, block = 961, 128, 4096, 128
    rng = np.random.default_rng(9)
    a, codes2, scales = _inputs(orc, rng, m, n, k, block, 2)
    w = smg.Q2Weights(codes2, scales, n, k, smg.Q2Params(block))
    ad = torch.from_numpy(a.view(np.int16)).cuda()
    out = [torch.zeros(m * n, dtype=torch.int16, device="cuda") for _ in range(2)]
    fn = smg.lib().smg_lowbit_matmul_dev_noalloc
    fn.argtypes = [C.c_size_t] + [C.c_void_p] * 5
    st = torch.cuda.current_stream().cuda_stream
    assert fn(m, w._h, out[0].data_ptr(), ad.data_ptr(), None, st) == 0
    smg.matmul_q2(ad, w, out[1], m)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
