"""The DMA-staged dense GEMM (gemm_dense): every tile of its rule, K tails,
strided operands and stores, against a float64 product of the same 16-bit
inputs. The result is rounded to 16 bits once from an f32 sum, so the bound is
half an ulp of the result plus the f32 sum's error (K products, each within
2^-24 of the running sum's magnitude), stated relative to 1 + |w|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one shape a tile: 256x256, 128x256, 64x128, 64x64 (twice), 32x64, ragged in m and
# n (test_host_logic.py holds the rule to them)
TILES = [(4000, 4090, 520), (500, 14300, 2056), (1000, 3001, 2056), (1000, 3001, 520), (250, 4001, 520),
         (61, 499, 520)]
# K edges on the smallest tile: one step, one chunk past it, one chunk short of
# two, whole steps
KS = [(33, 130, 64), (33, 130, 72), (33, 130, 120), (33, 130, 128), (5, 7, 1000)]


def _tol(k, bf16):
    return (2.0 ** -8 if bf16 else 2.0 ** -11) + k * 2.0 ** -24


def _mats(m, n, k, bf16, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.bfloat16 if bf16 else torch.float16
    a = torch.randn(m, k, generator=g, device="cuda").to(t)
    b = (torch.randn(k, n, generator=g, device="cuda") / k ** 0.5).to(t)
    return a, b


def _bits(x):
    import torch
    return x.contiguous().cpu().view(torch.int16).numpy().view(np.uint16)


def _check(got, want, k, bf16):
    import torch
    err = ((got.double() - want).abs() / (1 + want.abs())).max().item()
    assert err <= _tol(k, bf16), err
    assert bool(torch.isfinite(got).all())


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", TILES + KS)
def test_packed_product(smg, m, n, k, bf16):
    import torch
    a, b = _mats(m, n, k, bf16, m + n + k)
    p = (smg.prepack_bf16 if bf16 else smg.prepack_f16)(_bits(b), n, k)
    c = torch.empty(m, n, dtype=a.dtype, device="cuda")
    (smg.matmul_bf16_packed if bf16 else smg.matmul_f16_packed)(a, p, c, m)
    _check(c, a.double() @ b.double(), k, bf16)


@pytest.mark.parametrize("graph", ["bias", "scale_bias_relu", "interpreted"])
@pytest.mark.parametrize("m,n,k", TILES)
def test_packed_epilogue(smg, m, n, k, graph):
    """The compiled stores and the interpreted one on each tile (row-major and,
    interpreted, column-major C). beta 0.5 is exact in the store."""
    import torch
    a, b = _mats(m, n, k, False, 3)
    p = smg.prepack_f16(_bits(b), n, k)
    bias, scale = (torch.randn(n, device="cuda").half() for _ in range(2))
    row = torch.randn(m, device="cuda").half()
    h = (0.5 * (a.double() @ b.double())).half().double()  # the graph runs on the rounded product
    g = smg.Gemm(a, p, m).beta(0.5)
    c = torch.empty(m, n, dtype=torch.float16, device="cuda")
    if graph == "bias":
        g, want = g.add_col(bias), h + bias.double()
    elif graph == "scale_bias_relu":
        g, want = g.mul_col(scale).add_col(bias).relu(), (h * scale.double() + bias.double()).clamp(min=0)
    else:
        g, want = g.col_major_output().mul_row(row).add_col(bias), h * row.double()[:, None] + bias.double()
        c = torch.empty(n, m, dtype=torch.float16, device="cuda")
    g.run(c)
    got = c.t() if graph == "interpreted" else c
    # the product's rounding may fall to either side (one f16 ulp, scaled by
    # the largest |factor| drawn, below 5), then the store's own half ulp
    err = ((got.double() - want).abs() / (1 + want.abs() + 5 * h.abs())).max().item()
    assert err <= 2 * _tol(k, False), err


@pytest.mark.parametrize("alpha", [0.0, 0.75])
@pytest.mark.parametrize("bcol", [True, False])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", TILES[2:] + KS)
def test_strided_views(smg, m, n, k, bf16, bcol, alpha):
    """Views of larger arrays whose other elements are NaN (nothing outside a
    view is read into a sum), C a padded view; a column-major B is read in
    place, a row-major one packed."""
    import torch
    a, b = _mats(m, n, k, bf16, 7)
    lda, ldb, ldc = k + 8, (k if bcol else n) + 16, n + 3
    nan = lambda r, c: torch.full((r, c), float("nan"), dtype=a.dtype, device="cuda")  # noqa: E731
    av, bv, cv = nan(m, lda), nan(n if bcol else k, ldb), nan(m, ldc)
    av[:, :k] = a
    bv[:, :k if bcol else n] = b.t() if bcol else b
    c0 = torch.randn(m, n, device="cuda").to(a.dtype)
    if alpha:
        cv[:, :n] = c0
    f = smg.gemm_bf16 if bf16 else smg.gemm_f16
    f(m, n, k, cv, ldc, 1, av, lda, 1, bv, *((1, ldb) if bcol else (ldb, 1)), alpha, 1.0)
    want = a.double() @ b.double() + alpha * c0.double()
    _check(cv[:, :n], want, k, bf16)
    assert bool(cv[:, n:].isnan().all())  # the padding is untouched


def test_strided_result_may_share_memory_with_b(smg):
    """C over B's own memory (packing reads all of B first): the direct read
    stays off it."""
    import torch
    m = n = k = 256
    a, b = _mats(m, n, k, False, 11)
    bt = b.t().contiguous()
    want = a.double() @ b.double()
    smg.gemm_f16(m, n, k, bt, n, 1, a, k, 1, bt, 1, k, 0.0, 1.0)
    _check(bt, want, k, False)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", [(61, 499, 523), (1, 130, 7), (33, 65, 1), (300, 1001, 2049), (5, 9, 63)])
def test_products_over_any_k(smg, m, n, k, bf16):
    """K not a multiple of 8, unaligned rows and column strides: A packed on
    the device (host, device, packed and strided calls alike), NaN outside
    every view."""
    import torch
    a, b = _mats(m, n, k, bf16, m * k)
    want = a.double() @ b.double()
    p = (smg.prepack_bf16 if bf16 else smg.prepack_f16)(_bits(b), n, k)
    mul = smg.matmul_bf16_packed if bf16 else smg.matmul_f16_packed
    c = torch.empty(m, n, dtype=a.dtype, device="cuda")
    mul(a, p, c, m)
    _check(c, want, k, bf16)
    ch = np.zeros(m * n, np.uint16)
    mul(_bits(a).ravel(), p, ch, m)
    assert np.array_equal(ch, _bits(c).ravel())
    f = smg.gemm_bf16 if bf16 else smg.gemm_f16
    at = torch.full((k, 2 * m + 1), float("nan"), dtype=a.dtype, device="cuda")
    at[:, 1::2][:, :m] = a.t()  # A[i, l] at 1 + 2 i + l (2 m + 1)
    bt = torch.full((n, k + 1), float("nan"), dtype=a.dtype, device="cuda")
    bt[:, 1:] = b.t()
    c0 = torch.randn(m, n, device="cuda").to(a.dtype)
    c = c0.clone()
    f(m, n, k, c, n, 1, at.view(-1)[1:], 2, 2 * m + 1, bt.view(-1)[1:], 1, k + 1, 0.5, 1.0)
    _check(c, want + 0.5 * c0.double(), k, bf16)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("m,n,k", [(32, 300, 127), (32, 300, 129), (33, 300, 63), (33, 300, 65), (128, 128, 63),
                                   (129, 128, 63), (1, 1, 1)])
def test_strided_calls_with_and_without_a_packed(smg, m, n, k, bf16):
    """Both sides of the line up to which a strided call reads such an A where
    it is: the packed weights' call, which always packs it, gives the same
    bits."""
    import torch
    a, b = _mats(m, n, k, bf16, m + k)
    p = (smg.prepack_bf16 if bf16 else smg.prepack_f16)(_bits(b), n, k)
    c, e = (torch.empty(m, n, dtype=a.dtype, device="cuda") for _ in range(2))
    (smg.matmul_bf16_packed if bf16 else smg.matmul_f16_packed)(a, p, e, m)
    at = a.t().contiguous()
    (smg.gemm_bf16 if bf16 else smg.gemm_f16)(m, n, k, c, n, 1, at, 1, m, b, n, 1, 0.0, 1.0)
    _check(c, a.double() @ b.double(), k, bf16)
    assert torch.equal(c.view(torch.int16), e.view(torch.int16))


def test_odd_k_product_captured_without_scratch(smg):
    """A first odd-K product on a stream under capture allocates nothing (it
    reads A as it is) and replays right; eager calls on the stream then pack."""
    import torch
    m, n, k = 40, 200, 333
    a, b = _mats(m, n, k, False, 5)
    p = smg.prepack_f16(_bits(b), n, k)
    c, e = (torch.empty(m, n, dtype=a.dtype, device="cuda") for _ in range(2))
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        smg.matmul_f16_packed(a, p, c, m)
    for seed in (6, 7):
        a.copy_(_mats(m, n, k, False, seed)[0])
        g.replay()
        torch.cuda.synchronize()
        _check(c, a.double() @ b.double(), k, False)
        with torch.cuda.stream(s):
            smg.matmul_f16_packed(a, p, e, m)
        torch.cuda.synchronize()
        _check(e, a.double() @ b.double(), k, False)


def test_odd_k_graphs_hold_no_scratch(smg):
    """Two graphs captured on one stream after eager calls warmed it, replayed on
    two streams at once beside eager calls on the capture stream: each reads its
    own A (a packed copy in the stream's scratch would be overwritten by the
    others)."""
    import torch
    m, n, k = 1000, 500, 1001
    b = _mats(m, n, k, False, 5)[1]
    p = smg.prepack_f16(_bits(b), n, k)
    cap = torch.cuda.Stream()
    a = [_mats(m, n, k, False, 20 + i)[0] for i in range(3)]
    c = [torch.empty(m, n, dtype=torch.float16, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    with torch.cuda.stream(cap):
        smg.matmul_f16_packed(a[2], p, c[2], m)  # scratch of the largest size is there
    torch.cuda.synchronize()
    graphs = []
    for i in range(2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=cap):
            for _ in range(4):
                smg.matmul_f16_packed(a[i], p, c[i], m)
        graphs.append(g)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for rep in range(4):
        for i in range(3):
            a[i].copy_(_mats(m, n, k, False, 100 * rep + i)[0])
            c[i].fill_(float("nan"))
        torch.cuda.synchronize()
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                graphs[i].replay()
        with torch.cuda.stream(cap):
            for _ in range(4):
                smg.matmul_f16_packed(a[2], p, c[2], m)
        torch.cuda.synchronize()
        for i in range(3):
            _check(c[i], a[i].double() @ b.double(), k, False)


def test_odd_k_calls_of_several_threads_on_one_stream(smg):
    """Host threads that share a stream: a call's packing and product stay
    together, whatever the threads' sizes (the scratch grows between them)."""
    import threading
    import torch
    s = torch.cuda.Stream()
    jobs, err = [], []
    for t in range(4):
        m, n, k = 400 + 300 * t, 200, 1001 + 2 * t
        a, b = _mats(m, n, k, False, 60 + t)
        p = smg.prepack_f16(_bits(b), n, k)
        jobs.append((a, b, p, [torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda") for _ in range(24)]))
    torch.cuda.synchronize()

    def work(a, p, cs):
        try:
            with torch.cuda.stream(s):
                for c in cs:
                    smg.matmul_f16_packed(a, p, c, a.shape[0])
        except Exception as e:  # noqa: BLE001
            err.append(e)

    ts = [threading.Thread(target=work, args=(a, p, cs)) for a, b, p, cs in jobs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert not err, err
    for a, b, p, cs in jobs:
        want = a.double() @ b.double()
        for c in cs:
            _check(c, want, a.shape[1], False)


def test_odd_k_call_beside_another_threads_capture(smg):
    """An eager call that needs scratch for the first time on its stream, while
    this thread captures another stream in the default mode: neither the capture
    nor the call fails."""
    import threading
    import torch
    m, n, k = 2000, 96, 1003
    a, b = _mats(m, n, k, False, 70)
    p = smg.prepack_f16(_bits(b), n, k)
    other, cap = torch.cuda.Stream(), torch.cuda.Stream()
    c, d = (torch.empty(m, n, dtype=torch.float16, device="cuda") for _ in range(2))
    smg.matmul_f16_packed(a[:16].contiguous(), p, c[:16].contiguous(), 16)  # kernels are loaded
    torch.cuda.synchronize()
    err = []

    def call():
        try:
            with torch.cuda.stream(other):
                smg.matmul_f16_packed(a, p, c, m)
        except Exception as e:  # noqa: BLE001
            err.append(e)

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        smg.matmul_f16_packed(a, p, d, m)
        t = threading.Thread(target=call)
        t.start()
        t.join()
    assert not err, err
    want = a.double() @ b.double()
    for _ in range(2):
        d.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        _check(d, want, k, False)
    _check(c, want, k, False)


def test_odd_k_scratch_grows_beside_another_threads_capture(smg):
    """As above with a smaller buffer there already: outgrown, it is given back
    and replaced during the capture."""
    import threading
    import torch
    m, n, k = 2000, 96, 1003
    a, b = _mats(m, n, k, False, 71)
    p = smg.prepack_f16(_bits(b), n, k)
    other, cap = torch.cuda.Stream(), torch.cuda.Stream()
    c, d = (torch.empty(m, n, dtype=torch.float16, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        smg.matmul_f16_packed(a[:16], p, c[:16], 16)
    torch.cuda.synchronize()
    err = []

    def call():
        try:
            with torch.cuda.stream(other):
                smg.matmul_f16_packed(a, p, c, m)
        except Exception as e:  # noqa: BLE001
            err.append(e)

    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        smg.matmul_f16_packed(a, p, d, m)
        t = threading.Thread(target=call)
        t.start()
        t.join()
    assert not err, err
    d.fill_(float("nan"))
    g.replay()
    torch.cuda.synchronize()
    want = a.double() @ b.double()
    _check(d, want, k, False)
    _check(c, want, k, False)
