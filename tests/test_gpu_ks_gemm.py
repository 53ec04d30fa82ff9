"""GPU: the K-split block-scaled GEMM (MatMulBnb4 with float16 activations and
five or more rows; int8-activation MatMulNBits with many rows) at the edges of
its tiles: one and a few rows past a 32-row tile, columns past a wave's 32, K of
one pair of 64-code steps, of a half step and of uneven groups, every block
mode. MatMulBnb4 and the int8 path are compared with float64 at the bound of one
binary16 rounding plus float32 sums over K; infinities reach the sums as the
products do."""
import numpy as np
import pytest

from oracle import int8a as Q8
from oracle import oracle as O
from oracle import quant as Q

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def ops():
    from xrgpu_amd import ops as _ops
    return _ops


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def close(got, exact, mag, K, half):
    """One rounding of the result (2^-11 or 2^-24 of it), float32 sums and the
    codebook terms' 2^-22: K + 4 units of 2^-24 of the sum of magnitudes at most."""
    lim = np.abs(exact) * (2.0 ** -11 if half else 2.0 ** -24) + mag * ((K + 4) * 2.0 ** -24) + 2.0 ** -24
    err = np.abs(got.astype(np.float64) - exact)
    assert np.all(err <= lim), float((err - lim).max())


BNB = [  # M, K, N, block, quant_type
    (5, 32, 1, 32, 1),          # half a step
    (5, 96, 33, 32, 0),         # K not a multiple of 64
    (32, 128, 32, 64, 1),       # one pair of steps
    (33, 192, 65, 64, 0),       # second row tile of one row; K not a multiple of 128
    (64, 1024, 130, 128, 1),
    (97, 1152, 257, 128, 1),    # 18 steps
    (130, 2048, 100, 256, 0),
    (250, 4096, 512, 64, 1),
    (129, 1088, 2100, 32, 1),   # 17 steps over the groups
    (3, 14336, 40, 64, 1),      # rows that do not fit the GEMV's LDS
]


@pytest.mark.parametrize("M,K,N,bs,qt", BNB)
def test_bnb4(gpu, M, K, N, bs, qt):
    rng = np.random.default_rng(M + K + N + bs)
    a = rng.standard_normal((M, K)).astype(np.float16)
    b = rng.integers(0, 256, N * K // 2, dtype=np.uint8)
    s = rng.uniform(0.02, 1.5, N * K // bs).astype(np.float16)
    assert ops().bnb4_kernel(M, K, N, bs, qt, 1, torch.float16) == "bnb4_gemm"
    got = ops().matmul_bnb4(dev(a), dev(b), dev(s), K=K, N=N, block_size=bs, quant_type=qt).cpu().numpy()
    codes = np.stack((b >> 4, b & 15), -1).reshape(N, K)
    W = (Q.NF4 if qt == 1 else Q.FP4).astype(np.float64)[codes] * np.repeat(s.astype(np.float64).reshape(N, -1), bs, 1)
    close(got, a.astype(np.float64) @ W.T, np.abs(a).astype(np.float64) @ np.abs(W).T, K, True)


@pytest.mark.parametrize("qt", [1, 0])
def test_bnb4_nonfinite(gpu, qt):
    """An infinite or NaN activation gives what its products give: code by code."""
    M, K, N, bs = 6, 128, 16, 32
    a = np.ones((M, K), np.float16)
    a[1, 3], a[2, 70], a[3, 127], a[4, 0] = np.inf, -np.inf, np.nan, 65504
    b = np.zeros((N, K // 2), np.uint8)
    b[:] = (np.arange(N, dtype=np.uint8) * 17)[:, None]  # column n holds code n everywhere
    s = np.full(N * K // bs, 0.5, np.float16)
    got = ops().matmul_bnb4(dev(a), dev(b.reshape(-1)), dev(s), K=K, N=N, block_size=bs, quant_type=qt).cpu().numpy()
    ref = Q.matmul_bnb4(a, b.reshape(-1), s, K=K, N=N, block_size=bs, quant_type=qt)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fin = np.isfinite(ref)
    assert np.allclose(got[fin].astype(np.float64), ref[fin].astype(np.float64), rtol=2e-3, atol=1e-3)


@pytest.mark.parametrize("qt", [1, 0])
def test_bnb4_codebook_precision(gpu, qt):
    """Two products that nearly cancel show the codebook's own error: the weights are
    held to a quarter of float32's 2^-24 (a float32 table rounds to half of it), whose
    share in the difference is at most 0.5 units of 2^-24 of the magnitudes, beside the
    roundings of the scale and of the result."""
    book = (Q.NF4 if qt == 1 else Q.FP4).astype(np.float64)
    rows = []
    for c1 in range(16):
        for c2 in range(16):
            a1 = np.arange(1025, 2049, dtype=np.float64)
            if c1 == c2 or book[c1] == 0 or book[c2] == 0:
                continue
            a2 = -np.round(a1 * book[c1] / book[c2])
            ok = np.abs(a2) <= 2048  # exact in binary16
            if ok.any():
                i = np.abs(a1 * book[c1] + a2 * book[c2])[ok].argmin()
                rows.append((c1, c2, a1[ok][i], a2[ok][i]))
    M, K, bs = len(rows), 32, 32
    zero = 7 if qt == 1 else 0
    a, codes = np.zeros((M, K)), np.full((M, K), zero)
    for m, (c1, c2, a1, a2) in enumerate(rows):
        a[m, :2], codes[m, :2] = (a1, a2), (c1, c2)
    b = (codes[:, 0::2] << 4 | codes[:, 1::2]).astype(np.uint8)
    s = np.random.default_rng(qt).uniform(0.3, 1.7, M).astype(np.float16)
    assert ops().bnb4_kernel(M, K, M, bs, qt, 1, torch.float16) == "bnb4_gemm"
    got = np.diag(ops().matmul_bnb4(dev(a.astype(np.float16)), dev(b.reshape(-1)), dev(s), K=K, N=M, block_size=bs,
                                    quant_type=qt).cpu().numpy()).astype(np.float64)
    terms = a[:, :2] * book[codes[:, :2]] * s.astype(np.float64)[:, None]
    exact, mag = terms.sum(1), np.abs(terms).sum(1)
    lim = np.abs(exact) * (2.0 ** -11 + 2.0 ** -22) + mag * 0.5 * 2.0 ** -24 + 2.0 ** -25
    assert np.all(np.abs(got - exact) <= lim), float(((np.abs(got - exact) - np.abs(exact) * 2.0 ** -11) / mag).max() * 2 ** 24)


I8A = [  # M, K, N, block, zero points, bias, dtype
    (2049, 128, 1030, 32, True, True, np.float16),   # one pair of steps
    (33, 1024, 8200, 64, True, False, np.float32),
    (97, 1152, 2500, 128, True, True, np.float16),   # nine activation blocks over the groups
    (65, 2176, 2001, 32, False, True, np.float32),
    (8, 8192, 4100, 256, True, False, np.float16),
]


@pytest.mark.parametrize("M,K,N,bs,zp,bias,dt", I8A)
def test_int8a(gpu, M, K, N, bs, zp, bias, dt):
    assert M >= 8 and M * K * N >= 1 << 28  # the GEMM takes it
    rng = np.random.default_rng(M + K + N + bs)
    kb = K // bs
    A = (rng.standard_normal((M, K)) * rng.uniform(0.2, 4, (M, 1))).astype(dt)
    B = rng.integers(0, 256, (N, kb, bs // 2), dtype=np.uint8)
    S = rng.uniform(0.005, 0.05, (N, kb)).astype(dt)
    Z = rng.integers(0, 256, (N, (kb + 1) // 2), dtype=np.uint8) if zp else None
    b = (rng.standard_normal(N) * 0.1).astype(dt) if bias else None
    got = ops().matmul_nbits_int8a(dev(A), dev(B), dev(S), dev(Z), dev(b), K=K, N=N, block_size=bs).cpu().numpy()
    kind = O.ZP_PACKED if zp else None
    ref = Q8.matmul_nbits_int8a(A, B, S, Z, b, K=K, N=N, block_size=bs, zp_kind=kind, out_dtype=np.float64)
    q, sa = Q8.quantize_activations(A, K)
    W = O.dequantize(B, S, Z, K, 4, bs, kind).astype(np.float64)
    mag = np.abs(q.astype(np.float64) * np.repeat(sa.astype(np.float64), 128, 1)) @ np.abs(W).T
    close(got, ref, mag, K // 16, dt == np.float16)  # block sums are exact: a few roundings per block


@pytest.mark.parametrize("M", [7, 520])  # the GEMV, the GEMM (2^28 multiply-adds)
@pytest.mark.parametrize("bs,dt", [(32, np.float16), (128, np.float32)])
def test_int8a_nonfinite(gpu, M, bs, dt):
    """A block of 128 activations that holds an infinity or NaN has no scale: its row is
    NaN, as in the oracle (Inf times the other codes' zero), whatever the row count;
    the other rows are what they are without it."""
    K, N = 1024, 520
    assert (M >= 8 and M * K * N >= 1 << 28) == (M == 520)
    rng = np.random.default_rng(M + bs)
    A = rng.standard_normal((M, K)).astype(dt)
    B = rng.integers(0, 256, (N, K // bs, bs // 2), dtype=np.uint8)
    S = rng.uniform(0.005, 0.05, (N, K // bs)).astype(dt)
    bad = {0: (5, np.inf), 2: (700, -np.inf), 3: (130, np.nan), M - 1: (1023, np.inf)}
    clean = ops().matmul_nbits_int8a(dev(A), dev(B), dev(S), K=K, N=N, block_size=bs).cpu().numpy()
    A[2, 701] = np.inf
    for m, (k, v) in bad.items():
        A[m, k] = v
    A[1, 0:128:32] = np.inf  # one in every chunk of 32
    got = ops().matmul_nbits_int8a(dev(A), dev(B), dev(S), K=K, N=N, block_size=bs).cpu().numpy()
    rows = sorted({1, *bad})
    ref = Q8.matmul_nbits_int8a(A[rows], B, S, None, None, K=K, N=N, block_size=bs, zp_kind=None)
    assert np.isnan(ref).all() and np.isnan(got[rows]).all()
    rest = np.setdiff1d(np.arange(M), rows)
    assert np.array_equal(got[rest], clean[rest])


def test_bnb4_two_gib_of_activations(gpu):
    """Activations that end just below 2^31 bytes: the steps past the last row's K read
    zeros, not the first rows (whose infinities would reach the last row)."""
    M, K, N, bs = (1 << 25) - 1, 32, 8, 32
    rng = np.random.default_rng(1)
    b = dev(rng.integers(0, 256, N * K // 2, dtype=np.uint8))
    s = dev(rng.uniform(0.1, 1, N).astype(np.float16))
    A = torch.zeros((M, K), dtype=torch.float16, device="cuda")
    A[:64] = float("inf")
    A[-8:] = torch.randn(8, K, device="cuda", generator=torch.Generator("cuda").manual_seed(2)).half()
    assert ops().bnb4_kernel(M, K, N, bs, 1, 1, torch.float16) == "bnb4_gemm"
    y = ops().matmul_bnb4(A, b, s, K=K, N=N, block_size=bs)
    assert torch.equal(y[-8:], ops().matmul_bnb4(A[-8:].contiguous(), b, s, K=K, N=N, block_size=bs))
    assert torch.isfinite(y[64:]).all()


def off(a, items=1):
    """a on the GPU, contiguous, its data `items` elements past an allocation's start."""
    buf = torch.zeros(a.size + items, dtype=dev(a).dtype, device="cuda")
    buf[items:] = dev(a).flatten()
    return buf[items:].view(a.shape)


@pytest.mark.parametrize("bs", [32, 64])
def test_bnb4_unaligned_absmax(gpu, bs):
    """absmax two bytes past a word (the GEMM's word loads would be misaligned): the GEMV's
    results, row for row."""
    M, K, N = 9, 256, 96
    rng = np.random.default_rng(bs)
    a = dev(rng.standard_normal((M, K)).astype(np.float16))
    b = dev(rng.integers(0, 256, N * K // 2, dtype=np.uint8))
    s = rng.uniform(0.02, 1.5, N * K // bs).astype(np.float16)
    kw = dict(K=K, N=N, block_size=bs)
    got = ops().matmul_bnb4(a, b, off(s), **kw)
    # the same four-row passes, by calls of four rows (aligned absmax)
    want = torch.cat([ops().matmul_bnb4(torch.cat([a[m:m + 4], a[:4]])[:4].contiguous(), b, dev(s), **kw)[:M - m]
                      for m in range(0, M, 4)])
    assert torch.equal(got, want)


@pytest.mark.parametrize("which", ["scales", "zero_points"])
def test_int8a_unaligned_metadata(gpu, which):
    """Scales at an odd element or zero points at an odd byte: the GEMV's results."""
    M, K, N, bs = 264, 1024, 1000, 32
    assert M * K * N >= 1 << 28
    rng = np.random.default_rng(5)
    A = dev(rng.standard_normal((M, K)).astype(np.float16))
    B = dev(rng.integers(0, 256, (N, K // bs, bs // 2), dtype=np.uint8))
    S = rng.uniform(0.005, 0.05, (N, K // bs)).astype(np.float16)
    Z = rng.integers(0, 256, (N, K // bs // 2), dtype=np.uint8)
    kw = dict(K=K, N=N, block_size=bs)
    got = ops().matmul_nbits_int8a(A, B, off(S) if which == "scales" else dev(S), off(Z) if which == "zero_points" else dev(Z), **kw)
    want = torch.cat([ops().matmul_nbits_int8a(A[m:m + 6].contiguous(), B, dev(S), dev(Z), **kw) for m in range(0, M, 6)])
    assert torch.equal(got, want)
