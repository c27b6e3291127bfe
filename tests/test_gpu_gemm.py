"""The step-DMA MFMA GEMM (tinybrain_amd/csrc/tbh_gemm.h) at the edges of its
tiles, steps and plans, against a float64 product of the oracle's dequantized
weights.

The bound, per output of an x row and a weight column, in P = |x|_2 |w|_2:
rounding a sum of K products of random signs after each product (the MFMA adds
32 at a time, splits and pieces add a few sums) errs with a standard deviation
of 2^-24 / sqrt(3) * P / K * sqrt(1 + 2 + .. + K) <= 0.41 * 2^-24 P, whatever K;
the two f16 pieces that hold fp32 x and a runtime-layout weight to 2^-22 and
2^-21 of each element add under 0.3 * 2^-21 P / sqrt(K), 0.05 to 0.3 * 2^-24 P
here.  8 * 2^-24 P is over ten of these.  A product that loses the low piece of x
(2^-11 of each element: 2400 / sqrt(K) * 2^-24 P) is past it at every K the
kernel takes (test_f16_pieces.py)."""
import numpy as np
import pytest

import oracle as O
from tinybrain_amd._launches import gemms, launches
from tinybrain_amd import _abi
import tinybrain_amd as T
from test_gpu_sweep import _oracle_weight, _weight

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def backend():
    b = T.HIPBackend(0)
    yield b
    b.close()


BOUND = 8 * 2.0**-24


def _check(y, x, W, what):
    """y, x: torch tensors on the GPU; W: the oracle's [K, N] weight."""
    import torch

    x64, W64 = x.double(), torch.from_numpy(np.asarray(W, np.float64)).to(x.device)
    err = (y.double() - x64 @ W64).abs() / (x64.norm(dim=1)[:, None] * W64.norm(dim=0)[None, :])
    worst = float(err.max())
    assert worst <= BOUND, (what, worst / 2.0**-24)


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
        xb = xb.cuda()
        _check(backend.matmul_bf16_device(xb, w), xb, W, (kind, K, N, M, "bf16"))
        if M > 64:   # fp32 x: two f16 pieces
            x = torch.from_numpy(x).cuda()
            _check(backend.matmul_device(x, w), x, W, (kind, K, N, M, "fp32"))


def _tile_launches(backend, x, w, y):
    import torch

    stream = torch.cuda.Stream()
    f = backend.matmul_bf16_device if x.dtype == torch.bfloat16 else backend.matmul_device
    torch.cuda.synchronize()
    f(x, w, out=y, stream=stream)
    torch.cuda.synchronize()
    return launches(lambda: f(x, w, out=y, stream=stream), stream)


# every tile of every weight kind and form of x, (16-row tiles, 128-column
# tiles), with M, N and K off its edges: a product of a few K steps, and one
# whose K is split over all tiles ("split") or over the tiles of a last,
# part-filled round ("tail"); the plans are those for 256 CUs
TILES = [
    ("int8_zp", "bf16", 80, 123, 67, (4, 1), "whole"),
    ("int8", "bf16", 744, 101, 114, (4, 1), "split"),
    ("int8_zp", "bf16", 1744, 787, 2341, (4, 1), "tail"),
    ("int8", "bf16", 88, 6595, 569, (4, 2), "whole"),
    ("int8_zp", "bf16", 5144, 986, 1289, (4, 2), "split"),
    ("int8", "bf16", 72, 1435, 1353, (8, 1), "whole"),
    ("int8_zp", "bf16", 2904, 129, 2807, (8, 1), "split"),
    ("int8", "bf16", 2200, 2441, 1602, (8, 1), "tail"),
    ("int8_zp", "bf16", 96, 7114, 884, (8, 2), "whole"),
    ("int8", "bf16", 7032, 653, 2156, (8, 2), "split"),
    ("int8_zp", "bf16", 88, 1294, 2984, (12, 1), "whole"),
    ("int8", "bf16", 4968, 659, 1876, (12, 1), "split"),
    ("int8_zp", "bf16", 96, 3286, 2484, (12, 2), "whole"),
    ("int8", "bf16", 8080, 910, 2055, (12, 2), "split"),
    ("int8_zp", "bf16", 72, 3043, 1990, (16, 1), "whole"),
    ("int8", "bf16", 6320, 541, 2358, (16, 1), "split"),
    ("int8_zp", "bf16", 80, 8525, 1356, (16, 2), "whole"),
    ("int8", "bf16", 920, 6641, 2461, (16, 2), "tail"),
    ("int8_zp", "fp32", 88, 118, 126, (4, 1), "whole"),
    ("int8", "fp32", 648, 118, 83, (4, 1), "split"),
    ("int8_zp", "fp32", 1064, 782, 2333, (4, 1), "tail"),
    ("int8", "fp32", 80, 670, 2703, (4, 2), "whole"),
    ("int8_zp", "fp32", 1816, 145, 2806, (4, 2), "split"),
    ("int8", "fp32", 912, 1465, 2747, (4, 2), "tail"),
    ("int8_zp", "fp32", 160, 782, 2318, (8, 1), "whole"),
    ("int8", "fp32", 2520, 259, 2025, (8, 1), "split"),
    ("int8_zp", "fp32", 1176, 1835, 2303, (8, 1), "tail"),
    ("int8", "fp32", 104, 1561, 2563, (8, 2), "whole"),
    ("int8_zp", "fp32", 3512, 387, 2763, (8, 2), "split"),
    ("int8", "fp32", 560, 2771, 2967, (8, 2), "tail"),
    ("int4_nk_g32", "bf16", 96, 110, 82, (4, 1), "whole"),
    ("int4_nk_g32_zp", "bf16", 480, 121, 85, (4, 1), "split"),
    ("int4_nk_g32", "bf16", 608, 694, 2722, (4, 1), "tail"),
    ("int4_nk_g32_zp", "bf16", 160, 3013, 1311, (4, 2), "whole"),
    ("int4_nk_g32", "bf16", 2208, 399, 1593, (4, 2), "split"),
    ("int4_nk_g32_zp", "bf16", 992, 1494, 2745, (4, 2), "tail"),
    ("int4_nk_g32", "bf16", 96, 686, 2732, (8, 1), "whole"),
    ("int4_nk_g32_zp", "bf16", 1568, 171, 2707, (8, 1), "split"),
    ("int4_nk_g32", "bf16", 1120, 1458, 2761, (8, 1), "tail"),
    ("int4_nk_g32_zp", "bf16", 96, 2969, 2005, (8, 2), "whole"),
    ("int4_nk_g32", "bf16", 3936, 675, 1969, (8, 2), "split"),
    ("int4_nk_g32_zp", "bf16", 864, 3245, 2521, (8, 2), "tail"),
    ("int4_nk_g32", "bf16", 96, 1298, 2961, (12, 1), "whole"),
    ("int4_nk_g32_zp", "bf16", 2976, 421, 2725, (12, 1), "split"),
    ("int4_nk_g32", "bf16", 1632, 2551, 2337, (12, 1), "tail"),
    ("int4_nk_g32_zp", "bf16", 96, 3463, 2497, (12, 2), "whole"),
    ("int4_nk_g32", "bf16", 1312, 6561, 1869, (12, 2), "tail"),
    ("int4_nk_g32_zp", "bf16", 160, 3130, 2462, (16, 1), "whole"),
    ("int4_nk_g32", "bf16", 4064, 582, 2390, (16, 1), "split"),
    ("int4_nk_g32_zp", "bf16", 96, 8221, 1346, (16, 2), "whole"),
    ("int4_nk_g32", "bf16", 1120, 8259, 1989, (16, 2), "tail"),
    ("int4_nk_g32_zp", "fp32", 160, 105, 77, (4, 1), "whole"),
    ("int4_nk_g32", "fp32", 544, 111, 127, (4, 1), "split"),
    ("int4_nk_g32_zp", "fp32", 992, 658, 2741, (4, 1), "tail"),
    ("int4_nk_g32", "fp32", 160, 8841, 398, (4, 2), "whole"),
    ("int4_nk_g32_zp", "fp32", 2784, 646, 1059, (4, 2), "split"),
    ("int4_nk_g32", "fp32", 96, 665, 2954, (8, 1), "whole"),
    ("int4_nk_g32_zp", "fp32", 1440, 182, 2783, (8, 1), "split"),
    ("int4_nk_g32", "fp32", 1504, 1298, 2952, (8, 1), "tail"),
    ("int4_nk_g32_zp", "fp32", 96, 2350, 2565, (8, 2), "whole"),
    ("int4_nk_g32", "fp32", 2080, 899, 2242, (8, 2), "split"),
    ("int4_nk_g32_zp", "fp32", 608, 2701, 2982, (8, 2), "tail"),
    ("int4_nk_g32", "fp32", 96, 1294, 2993, (12, 1), "whole"),
    ("int4_nk_g32_zp", "fp32", 2272, 399, 2918, (12, 1), "split"),
    ("int4_kn_g32", "bf16", 88, 96, 74, (4, 1), "whole"),
    ("int4_kn_g32", "bf16", 456, 96, 65, (4, 1), "split"),
    ("int4_kn_g32", "bf16", 1784, 704, 2726, (4, 1), "tail"),
    ("int4_kn_g32", "bf16", 80, 704, 2728, (8, 1), "whole"),
    ("int4_kn_g32", "bf16", 904, 160, 2957, (8, 1), "split"),
    ("int4_kn_g32", "bf16", 2296, 1568, 2517, (8, 1), "tail"),
    ("int4_kn_g32", "bf16", 96, 8800, 780, (8, 2), "whole"),
    ("int4_kn_g32", "bf16", 6048, 4160, 275, (8, 2), "split"),
    ("int4_kn_g32", "bf16", 88, 1344, 2953, (12, 1), "whole"),
    ("int4_kn_g32", "bf16", 2136, 288, 2907, (12, 1), "split"),
    ("int4_kn_g32", "bf16", 72, 6720, 792, (16, 1), "whole"),
    ("int4_kn_g32", "bf16", 1888, 672, 2843, (16, 1), "split"),
    ("int4_kn_g32", "bf16", 664, 3008, 2785, (16, 1), "tail"),
    ("int4_kn_g32", "fp32", 80, 96, 88, (4, 1), "whole"),
    ("int4_kn_g32", "fp32", 400, 96, 101, (4, 1), "split"),
    ("int4_kn_g32", "fp32", 904, 704, 2712, (4, 1), "tail"),
    ("int4_kn_g32", "fp32", 72, 3072, 1330, (4, 2), "whole"),
    ("int4_kn_g32", "fp32", 1720, 960, 1304, (4, 2), "split"),
    ("int4_kn_g32", "fp32", 80, 704, 2860, (8, 1), "whole"),
    ("int4_kn_g32", "fp32", 1032, 160, 2727, (8, 1), "split"),
    ("int4_kn_g32", "fp32", 488, 1344, 2953, (8, 1), "tail"),
    ("int4_kn_g32", "fp32", 72, 1376, 2948, (8, 2), "whole"),
    ("int4_kn_g32", "fp32", 2200, 480, 2715, (8, 2), "split"),
    ("int4_kn_g32", "fp32", 776, 2720, 2956, (8, 2), "tail"),
]


@pytest.mark.parametrize("kind,form,K,N,M,tile,plan", TILES)
def test_tiles(backend, kind, form, K, N, M, tile, plan):
    import torch

    qt, pq = _weight(kind, K, N, seed=K + 5 * N)
    w = T.DeviceWeight(backend, pq)
    x = torch.from_numpy(O.fill_normal(13 * K + M, M * K).reshape(M, K)).cuda()
    if form == "bf16":
        x = x.to(torch.bfloat16)
    y = torch.empty((M, N), device="cuda")
    ls = _tile_launches(backend, x, w, y)
    if backend.cu_count == 256:
        assert [(g.tm, g.tn) for g in gemms(ls)] == [tile], ls
        assert ls[-1].name == {"whole": "gemm", "split": "split_sum", "tail": "tail_sum"}[plan], ls
    _check(y, x, _oracle_weight(qt, pq.layout), (kind, form, K, N, M))
    w.close()


# fp32 x up to 64 rows as three exact bf16 pieces, on weights past the rule's
# lines: INT8 from 32 Mi elements, INT4 from 10 Mi (17 rows) and from 32 Mi (12)
@pytest.mark.parametrize("kind,K,N", [
    ("int8", 8200, 4100),            # 64 x 256 tiles, split; 64 x 128 at 64 rows
    ("int4_nk_g32", 2080, 5133),     # 64 x 128 tiles, split
    ("int4_nk_g128", 8192, 4098),    # 64 x 256 tiles, split
    ("int8_zp", 1032, 33003),        # 64 x 128 tiles, a tail
])
def test_few_rows(backend, kind, K, N):
    import torch

    qt, pq = _weight(kind, K, N, seed=K + N)
    W = _oracle_weight(qt, pq.layout)
    w = backend.weight(pq)
    for M in (12, 16, 17, 33, 64):
        x = torch.from_numpy(O.fill_normal(19 * K + M, M * K).reshape(M, K)).cuda()
        _check(backend.matmul_device(x, w), x, W, (kind, K, N, M))


@pytest.mark.parametrize("kind,K,N,M", [
    ("int8", 2048, 256, 300),          # splits over all tiles
    ("int4_nk_g32", 4096, 384, 130),
    ("int4_kn_g32", 2048, 256, 260),
    ("int8", 512, 2560, 2100),         # whole
    ("int8", 1064, 782, 2333),         # tails of 64 x 128, 128 x 256 and 128 x 128 tiles
    ("int8_zp", 560, 2771, 2967),
    ("int4_nk_g32", 1504, 1298, 2952),
    ("int4_kn_g32", 488, 1344, 2953),
])
def test_small_scratch_same_bits(backend, kind, K, N, M):
    """Scratch that does not hold the pieces and partial tiles at once: rows and
    K parts one after the other, the same results bit for bit."""
    import torch

    qt, pq = _weight(kind, K, N, seed=5 * K + N)
    w = backend.weight(pq)
    x = torch.from_numpy(O.fill_normal(23 * K + M, M * K).reshape(M, K)).cuda()
    ref = torch.empty((M, N), device="cuda")
    ls = _tile_launches(backend, x, w, ref)
    if backend.cu_count == 256:
        assert ls[-1].name == ("tail_sum" if M > 2200 else "gemm" if M == 2100 else "split_sum"), ls
    for limit in (0, 1 << 20, 16 * (4 + 4 * ((K + 63) // 64 * 64)) + 600):
        backend.set_option(_abi.OPT_NOALLOC_SCRATCH_BYTES, limit)
        try:
            y = backend.matmul_device_noalloc(x, w, out=torch.empty_like(ref))
            torch.cuda.synchronize()
        finally:
            backend.set_option(_abi.OPT_NOALLOC_SCRATCH_BYTES, 0)
        assert torch.equal(y.view(torch.int32), ref.view(torch.int32)), (kind, K, N, M, limit)
    _check(ref, x, _oracle_weight(qt, pq.layout), (kind, K, N, M))


@pytest.mark.parametrize("kind", ["int8", "int4_nk_g32_zp"])
def test_rows_too_long(backend, kind):
    """K from 2^20 runs on the register-staged GEMM (buffer offsets of the other
    would pass 2^30)."""
    import torch

    K, N, M = 1 << 20, 24, 3
    qt, pq = _weight(kind, K, N, seed=11)
    w, W = T.DeviceWeight(backend, pq), _oracle_weight(qt, pq.layout)
    x, y = torch.from_numpy(O.fill_normal(31, M * K).reshape(M, K)).cuda(), torch.empty((M, N), device="cuda")
    for xi in (x, x.to(torch.bfloat16)):
        assert _tile_launches(backend, xi, w, y)[0].name == "gemm_bf16"
        _check(y, xi, W, (kind, K, N, M, xi.dtype))
    w.close()


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
    _check(y, x, _oracle_weight(qt, pq.layout), (kind, K, N, M))
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
