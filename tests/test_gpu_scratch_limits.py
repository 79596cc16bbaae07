"""Calls whose faster form needs scratch that cannot be had still run: the
allocations past a size fail (SMG_TEST_FAIL_ALLOC=N) as on a full device, and
each call takes the form that needs less, the same result as with memory."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bits(x):
    import torch
    return x.contiguous().cpu().view(torch.int16).numpy().view(np.uint16)


def _fresh(fn, stream=None):
    """fn on a thread of its own (host calls then have no staging buffer yet)."""
    import torch
    out, err = [], []

    def run():
        try:
            with torch.cuda.stream(stream or torch.cuda.default_stream()):
                out.append(fn())
        except Exception as e:  # noqa: BLE001
            err.append(e)

    t = threading.Thread(target=run)
    t.start()
    t.join()
    torch.cuda.synchronize()
    assert not err, err
    return out[0]


def test_odd_k_product_without_room_for_a(smg, monkeypatch):
    """A's packed copy (2.1 MB) past the limit, B's pack and the staging of A and
    C within it: device and host calls, packed and strided."""
    import torch
    m, n, k = 1000, 8, 1001
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randn(m, k, generator=g, device="cuda").half()
    b = (torch.randn(k, n, generator=g, device="cuda") / k ** 0.5).half()
    p = smg.prepack_f16(_bits(b), n, k)
    want = torch.empty(m, n, dtype=torch.float16, device="cuda")
    smg.matmul_f16_packed(a, p, want, m)
    ah, bh = _bits(a).ravel(), _bits(b).ravel()
    c, d = (torch.empty(m, n, dtype=torch.float16, device="cuda") for _ in range(2))
    ch, dh = (np.zeros(m * n, np.uint16) for _ in range(2))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    monkeypatch.setenv("SMG_TEST_FAIL_ALLOC", str(2 << 20))
    _fresh(lambda: smg.matmul_f16_packed(a, p, c, m), s)
    _fresh(lambda: smg.gemm_f16(m, n, k, d, n, 1, a, k, 1, b, n, 1, 0.0, 1.0), s)
    monkeypatch.setenv("SMG_TEST_FAIL_ALLOC", str(3 << 20))
    _fresh(lambda: smg.matmul_f16_packed(ah, p, ch, m))
    _fresh(lambda: smg.gemm_f16(m, n, k, dh, n, 1, ah, k, 1, bh, n, 1, 0.0, 1.0))
    monkeypatch.delenv("SMG_TEST_FAIL_ALLOC")
    for got in (_bits(c).ravel(), _bits(d).ravel(), ch, dh):
        assert np.array_equal(got, _bits(want).ravel())


def test_low_bit_call_without_room_for_the_gemm(smg, monkeypatch):
    """The many-row GEMM's rows (in whole tiles, K in whole steps) past a limit
    that the GEMV's fit in: device and host calls."""
    import torch
    m, n, k, block = 241, 320, 3968, 128
    rng = np.random.default_rng(2)
    codes = rng.integers(0, 256, k * n // 4, dtype=np.uint8)
    scales = rng.uniform(0.01, 0.05, n * k // block).astype(np.float16).view(np.uint16)
    w = smg.Q2Weights(codes, scales, n, k, smg.Q2Params(block))
    ah = rng.standard_normal(m * k).astype(np.float16).view(np.uint16)
    a = torch.from_numpy(ah.view(np.int16)).cuda()
    want, c = (torch.zeros(m * n, dtype=torch.int16, device="cuda") for _ in range(2))
    smg.matmul_q2(a, w, want, m)
    ch = np.zeros(m * n, np.uint16)
    torch.cuda.synchronize()
    monkeypatch.setenv("SMG_TEST_FAIL_ALLOC", str(3 << 19))
    _fresh(lambda: smg.matmul_q2(a, w, c, m), torch.cuda.Stream())
    # staging: A and C (2.0 MB) and the GEMV's rows (1.0 MB) fit in 3 MiB
    monkeypatch.setenv("SMG_TEST_FAIL_ALLOC", str(3 << 20))
    _fresh(lambda: smg.matmul_q2(ah, w, ch, m))
    monkeypatch.delenv("SMG_TEST_FAIL_ALLOC")
    assert torch.equal(c, want)
    assert np.array_equal(ch, _bits(want))
