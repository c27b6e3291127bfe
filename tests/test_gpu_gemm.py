"""The step-DMA MFMA GEMM (tinybrain_amd/csrc/tbh_gemm.h) at the edges of its
tiles, steps and plans, against a float64 product of the oracle's dequantized
weights.

The bound is derived, per output: S = (|x| |W|) is the sum of magnitudes that
the products and their partial sums stay under, so fp32 accumulation of K
products in 32-deep MFMA steps, at most 32 splits and the scalings err by at
most (K + 64) 2^-24 S; the two f16 pieces of fp32 x hold it to 2^-21 of the
row's largest element, and those of a runtime-layout weight hold it to 2^-21
of itself: 2^-20 S + 2^-21 max|x| (1 |W|).
"""
import numpy as np
import pytest

import oracle as O
from launches import gemms, launches
from tinybrain_amd import _abi
import tinybrain_amd as T
from test_gpu_sweep import _oracle_weight, _weight

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def backend():
    b = T.HIPBackend(0)
    yield b
    b.close()


def _check(y, x, W, what):
    x64, W64 = x.astype(np.float64), W.astype(np.float64)
    S = np.abs(x64) @ np.abs(W64)
    bound = ((x.shape[1] + 64) * 2.0**-24 + 2.0**-20) * S
    bound += 2.0**-21 * np.abs(x64).max(axis=1, keepdims=True) * np.abs(W64).sum(axis=0)
    worst = np.max(np.abs(y.astype(np.float64) - x64 @ W64) - bound)
    assert worst <= 0, (what, worst)


# K off the 64-deep step (one 8-wide piece, half a step, a step and a bit) and
# on it; N off the 16-, 128- and 256-column tiles and off 4 (scalar stores);
# groups of one, two and three chunks, four, and a whole row; N-blocks of 16,
# 32 and 64 rows.
CASES = [
    ("int8", 72, 1),
    ("int8", 1032, 130),
    ("int8", 2048, 255),
    ("int8_zp", 584, 129),
    ("int4_nk_g32", 96, 17),
    ("int4_nk_g32", 2048, 257),
    ("int4_nk_g64", 1088, 127),
    ("int4_nk_g96", 960, 130),
    ("int4_nk_g128", 4096, 100),
    ("int4_nk_g512", 512, 384),
    ("int4_nk_g32_zp", 608, 129),
    ("int4_kn_g16", 520, 80),
    ("int4_kn_g32", 1032, 160),
    ("int4_kn_g64", 2048, 320),
]


@pytest.mark.parametrize("kind,K,N", CASES)
def test_tile_edges(backend, kind, K, N):
    import torch

    qt, pq = _weight(kind, K, N, seed=K + 3 * N)
    W = _oracle_weight(qt, pq.layout)
    w = backend.weight(pq)
    for M in (1, 15, 63, 64, 65, 127, 129, 193, 257, 321):
        x = O.fill_normal(17 * K + M, M * K).reshape(M, K)
        xb = torch.from_numpy(x).to(torch.bfloat16)
        y = backend.matmul_bf16_device(xb.cuda(), w)
        torch.cuda.synchronize()
        _check(y.cpu().numpy(), xb.float().numpy(), W, (kind, K, N, M, "bf16"))
        if M > 64:   # fp32 x: two f16 pieces
            y = backend.matmul_device(torch.from_numpy(x).cuda(), w)
            torch.cuda.synchronize()
            _check(y.cpu().numpy(), x, W, (kind, K, N, M, "fp32"))


# fp32 x up to 64 rows as three exact bf16 pieces, on weights past the rule's
# lines: INT8 from 32 Mi elements, INT4 from 10 Mi (17 rows) and from 32 Mi (12)
@pytest.mark.parametrize("kind,K,N", [("int8", 8200, 4100), ("int4_nk_g32", 2080, 5133), ("int4_nk_g128", 8192, 4098)])
def test_few_rows(backend, kind, K, N):
    import torch

    qt, pq = _weight(kind, K, N, seed=K + N)
    W = _oracle_weight(qt, pq.layout)
    w = backend.weight(pq)
    for M in (12, 16, 17, 33, 64):
        x = O.fill_normal(19 * K + M, M * K).reshape(M, K)
        y = backend.matmul_device(torch.from_numpy(x).cuda(), w)
        torch.cuda.synchronize()
        _check(y.cpu().numpy(), x, W, (kind, K, N, M))


@pytest.mark.parametrize("kind,K,N,M", [
    ("int8", 2048, 256, 300),          # splits over all tiles
    ("int4_nk_g32", 4096, 384, 130),
    ("int4_kn_g32", 2048, 256, 260),
    ("int8", 512, 2560, 2100),         # more tiles than CUs: a tail split or whole rounds
])
def test_small_scratch_same_bits(backend, kind, K, N, M):
    """Scratch that does not hold the pieces and partial tiles at once: rows and
    K parts one after the other, the same results bit for bit."""
    import torch

    qt, pq = _weight(kind, K, N, seed=5 * K + N)
    w = backend.weight(pq)
    x = torch.from_numpy(O.fill_normal(23 * K + M, M * K).reshape(M, K)).cuda()
    ref = backend.matmul_device(x, w)
    torch.cuda.synchronize()
    for limit in (0, 1 << 20, 16 * (4 + 4 * ((K + 63) // 64 * 64)) + 600):
        backend.set_option(_abi.OPT_NOALLOC_SCRATCH_BYTES, limit)
        try:
            y = backend.matmul_device_noalloc(x, w, out=torch.empty_like(ref))
            torch.cuda.synchronize()
        finally:
            backend.set_option(_abi.OPT_NOALLOC_SCRATCH_BYTES, 0)
        assert torch.equal(y.view(torch.int32), ref.view(torch.int32)), (kind, K, N, M, limit)
    _check(ref.cpu().numpy(), x.cpu().numpy(), _oracle_weight(qt, pq.layout), (kind, K, N, M))


# fp32 x of long prompts, whose pieces pass 128 MiB and are made in parts: 4096
# rows at K = 8192, 3008 at K = 11008
@pytest.mark.parametrize("kind,K,M", [
    ("int4_kn_g32", 8192, 4033),
    ("int4_kn_g32", 8192, 4096),
    ("int4_kn_g32", 8192, 4097),
    ("int4_kn_g32", 11008, 3072),
    ("int8", 8192, 4160),
    ("int4_nk_g32", 8192, 4033),
    ("int4_nk_g32", 8192, 4100),
])
def test_pieces_in_parts(backend, kind, K, M):
    import torch

    N = 64
    qt, pq = _weight(kind, K, N, seed=K + M)
    w = backend.weight(pq)
    x = torch.from_numpy(O.fill_normal(29 * K + M, M * K).reshape(M, K)).cuda()
    y, stream = torch.empty((M, N), device="cuda"), torch.cuda.Stream()
    torch.cuda.synchronize()
    backend.matmul_device(x, w, out=y, stream=stream)
    torch.cuda.synchronize()
    ls = launches(lambda: backend.matmul_device(x, w, out=y, stream=stream), stream)
    # every part on the GEMM, in one form, with at most the pieces before it and
    # a sum after it
    assert {n for n, _, _ in ls} <= {"x_pieces", "gemm", "split_sum", "tail_sum"}, ls
    assert {g.pieces for g in gemms(ls)} == {2}, ls
    most = (128 << 20) // (64 * 4 * (-(-K // 64) * 64)) * 64
    assert len(gemms(ls)) == -(-M // most) and len(ls) <= 3 * len(gemms(ls)), ls
    _check(y.cpu().numpy(), x.cpu().numpy(), _oracle_weight(qt, pq.layout), (kind, K, N, M))
    z = backend.matmul_device_noalloc(x, w, out=torch.empty_like(y))
    torch.cuda.synchronize()
    assert torch.equal(z.view(torch.int32), y.view(torch.int32))


def _kernels(backend, kind, K, N, M, bf16):
    """Names of the kernels of one call on a weight of random bytes, the last
    stretch of them (its GEMM, or the last GEMV launch)."""
    import torch

    rng = np.random.default_rng(K + N)
    if kind == "int8":
        pq = T.QuantizedTensor((K, N), rng.integers(-127, 128, K * N, dtype=np.int8), np.full(N, 0.01, np.float32),
                               T.QuantizationMode.perChannel)
    else:
        pq = T.QuantizedTensor((K, N), rng.integers(-128, 128, K * N // 2, dtype=np.int8),
                               np.full(K * N // 32, 0.01, np.float32), T.QuantizationMode.int4,
                               T.QuantizationPrecision.int4, 32, None, T.Layout.NK_FLAT)
    w = T.DeviceWeight(backend, pq)
    x = torch.zeros((M, K), dtype=torch.bfloat16 if bf16 else torch.float32, device="cuda")
    y, stream = torch.empty((M, N), device="cuda"), torch.cuda.Stream()
    call = lambda: (backend.matmul_bf16_device if bf16 else backend.matmul_device)(x, w, out=y, stream=stream)
    torch.cuda.synchronize()
    call()                                                # its workspace
    torch.cuda.synchronize()
    names = {n for n, _, _ in launches(call, stream)}
    w.close()
    return names


# few rows of fp32 x on INT8 weights from 32 Mi elements: the GEMM from five
# rows, from four where K is 8192 or more (mfma_min_rows)
@pytest.mark.parametrize("K,N,M,gemv", [(2560, 14336, 4, True), (2560, 14336, 5, False), (6000, 6000, 4, True),
                                        (8704, 4096, 4, False)])
def test_few_rows_kernel(backend, K, N, M, gemv):
    names = _kernels(backend, "int8", K, N, M, False)
    assert any(n.startswith("gemv") for n in names) == gemv, names
    assert any(n in ("gemm", "gemm_bf16") for n in names) != gemv, names


# bf16 x on INT4 K-groups of a long K: tiles of 128 x 128 that fill the CUs in
# eight, four or (K below 4608) two parts stay on gemm_bf16 (keep_gemm_bf16)
@pytest.mark.parametrize("K,N,M,kept", [(4096, 4096, 512, True), (4128, 1020, 2047, True), (4800, 1024, 2048, False),
                                        (5632, 2048, 512, True), (8192, 1024, 512, True), (4096, 4096, 1024, False)])
def test_kept_kernel(backend, K, N, M, kept):
    names = _kernels(backend, "int4", K, N, M, True)
    if backend.cu_count == 256:
        assert ("gemm_bf16" in names, "gemm" in names) == (kept, not kept), names
