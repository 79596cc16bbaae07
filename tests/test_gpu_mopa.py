"""The DMA-staged f16 GEMM over 2-bit / 1-bit weights (gemm_mopa): both tiles, K
and column tails, block sizes, an epilogue."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -11  # f16: half an ulp relative


@pytest.fixture(scope="module")
def smg():
    import smegemm
    return smegemm


def _weights(smg, bits, n, k, block, seed):
    """Weights and the f16 matrix they stand for, rounded once a value."""
    rng = np.random.default_rng(seed)
    nb = (k + block - 1) // block
    scales = (rng.uniform(0.25, 1.0, (n, nb)) * rng.choice([-1.0, 1.0], (n, nb))).astype(np.float16)
    if bits == 1:
        bit = rng.integers(0, 2, (n, k), dtype=np.uint8)
        vals = 2 * bit.astype(np.float32) - 1
        packed = np.packbits(bit.ravel(), bitorder="little")
        w = smg.Q1Weights(packed, scales.view(np.uint16).ravel(), smg.WeightLayout.OutIn, n, k, block)
    else:
        book = np.array([-127, -31, 0, 90], np.float32)
        p = smg.Q2Params(block).with_codebook(book)
        code = rng.integers(0, 4, (n, k), dtype=np.uint8)
        vals = book[code]
        flat = np.concatenate([code.T.ravel(), np.zeros(-code.size % 4, np.uint8)]).reshape(-1, 4)  # depth by depth
        w = smg.Q2Weights((flat << np.array([0, 2, 4, 6], np.uint8)).sum(1, dtype=np.uint8),
                          scales.view(np.uint16).ravel(), n, k, p)
    sc = np.repeat(scales.astype(np.float32), block, axis=1)[:, :k]
    return w, (sc * vals).astype(np.float16)


# rows x columns that reach 128-row tiles (1-bit) and 256-row ones (both kinds:
# more than one pass of the chip's units with the smaller tiles)
SHAPES = [
    (1, 129, 1, 64, 64), (1, 200, 300, 200, 128), (1, 257, 129, 520, 64), (1, 385, 1000, 584, 256),
    (1, 2049, 4097, 136, 128), (2, 2049, 4097, 136, 128), (2, 2300, 4000, 328, 64), (2, 4096, 4096, 64, 256)]


@pytest.mark.parametrize("bits,m,n,k,block", SHAPES)
@pytest.mark.parametrize("ep", [False, True])
def test_mopa_gemm(smg, bits, m, n, k, block, ep):
    import torch
    w, wf = _weights(smg, bits, n, k, block, m + n + k)
    g = torch.Generator(device="cuda").manual_seed(k)
    a = torch.randn(m, k, device="cuda", generator=g).half()
    e = smg.Epilogue()
    bias = torch.randn(n, device="cuda", generator=g).half()
    if ep:
        e = smg.Epilogue().add_col(bias)
    c = torch.empty(m, n, dtype=torch.float16, device="cuda")
    (smg.matmul_q1_mopa_ep if bits == 1 else smg.matmul_q2_mopa_ep)(a, w, c, m, e)
    ad, wd = a.double(), torch.from_numpy(wf).cuda().double()
    prod = ad @ wd.t().contiguous()
    mag = ad.abs() @ wd.abs().t().contiguous()
    # f32 sums of exact products: k roundings of partial sums no larger than
    # mag; then the product and the epilogue's sum each rounded to f16
    tol = mag * k * 2.0 ** -24 + 2 * EPS * (prod.abs() + (bias.abs().double() if ep else 0)) + 2.0 ** -24
    want = prod + (bias.double() if ep else 0)
    assert ((c.double() - want).abs() <= tol).all()
