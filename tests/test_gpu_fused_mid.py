"""GPU: Qkv / Mlp on the 128-row tiles (normalised rows in a workspace, too few
256 x 256 tiles for the large pipeline) against the oracle at the edges: a last
row tile of one row, columns past a tile, K of one step, of an odd number of
steps (uneven K groups) and with a last block that is not whole, narrow and wide
tiles, every zero-point kind. Binary16 bar: max|d| <= 1e-2 max|Y|."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def ops():
    from xrgpu_amd import ops as _ops
    return _ops


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def weights(rng, N, K, bs, zp):
    kb = (K + bs - 1) // bs
    B = rng.integers(0, 256, (N, kb, bs // 2), dtype=np.uint8)
    S = rng.uniform(0.001, 0.02, (N, kb)).astype(np.float16)
    Z = None
    if zp == "packed":
        Z = rng.integers(0, 256, (N, (kb + 1) // 2), dtype=np.uint8)
    elif zp is not None:
        Z = rng.uniform(4, 12, (N, kb)).astype(np.float32 if zp == "float32" else np.float16)
    return B, S, Z


CASES = [  # M, K, N, Nkv, block, zero points, skip
    (65, 64, 40, 8, 32, None, True),        # one step: the second K group has none
    (129, 192, 130, 64, 32, "packed", False),  # three steps, a row tile of one row
    (100, 1000, 257, 65, 64, "float", True),   # a last block that is not whole
    (128, 2048, 512, 128, 128, None, False),
    (385, 320, 9000, 136, 64, "packed", True),  # past one round of narrow tiles: wide ones
    (257, 96, 11500, 64, 32, "float", False),
]
# past one round of narrow tiles, too few 256 x 256 ones: the wide form
WIDE_QKV = [(385, 128, 9000, 136, 32, None, False), (300, 320, 12001, 40, 64, "float32", True)]
WIDE_MLP = [
    (333, 192, 5632, 0, 32, None, True),
    (257, 96, 5500, 0, 32, "packed", False),   # a row tile of one row, a column tile not whole
    (256, 320, 11001, 0, 64, "float", True),   # odd width, five steps
    (300, 136, 6000, 0, 64, "float32", False),  # a last block that is not whole
]


def form(op, M, N, Nkv):
    """The tiles the dispatch picks for normalised rows and blocks of 32 and more (the
    family's name, gemm_q4_fused, also covers the 128 x 128 kernel that has no workspace)."""
    def up(a, b):
        return -(-a // b)

    def cols(w):
        return up(N, w // 2) if op == "mlp" else up(N, w) + 2 * up(Nkv, w)
    if M >= 128 and up(M, 256) * cols(256) >= 128:
        return "big"
    return "narrow" if up(M, 128) * cols(128) <= torch.cuda.get_device_properties(0).multi_processor_count else "wide"


def test_forms(gpu):
    """The cases below reach every form they are meant for."""
    for op, wide in (("qkv", WIDE_QKV), ("mlp", WIDE_MLP)):
        assert {form(op, *c[:1], *c[2:4]) for c in wide} == {"wide"}
        for M, K, N, Nkv, bs, zp, skip in wide:
            assert ops().fused_workspace_bytes(op, M, K, N, Nkv, block_size=bs, skip=skip) > 0
            if op == "mlp":  # (the query takes one width, Qkv has two)
                assert ops().select_kernel("MatMulNBitsMlp", M, K, N, 4, bs) == "gemm_q4_fused"
    assert {form("qkv", *c[:1], *c[2:4]) for c in CASES} == {"narrow", "wide"}
    assert {form("mlp", *c[:1], *c[2:4]) for c in CASES} == {"narrow", "big"}


@pytest.mark.parametrize("M,K,N,Nkv,bs,zp,skip", CASES + WIDE_QKV)
def test_qkv(gpu, M, K, N, Nkv, bs, zp, skip):
    rng = np.random.default_rng(M + K + N)
    A = rng.standard_normal((M, K)).astype(np.float16)
    sk = rng.standard_normal((M, K)).astype(np.float16) if skip else None
    g = rng.uniform(0.5, 1.5, K).astype(np.float16)
    q, k, v = (weights(rng, n, K, bs, zp) for n in (N, Nkv, Nkv))
    kw = dict(q_zero_points=q[2], k_zero_points=k[2], v_zero_points=v[2])
    got = ops().matmul_nbits_qkv(dev(A), dev(q[0]), dev(q[1]), dev(k[0]), dev(k[1]), dev(v[0]), dev(v[1]),
                                 norm_scale=dev(g), skip=dev(sk), block_size=bs, **{n: dev(z) for n, z in kw.items()})
    x = A.astype(np.float64) + (sk.astype(np.float64) if skip else 0)
    x = (x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-6) * g.astype(np.float64)).astype(np.float16)
    for y, w, n in zip(got[:3], (q, k, v), (N, Nkv, Nkv)):
        ref = O.matmul_nbits(x, w[0], w[1], w[2], None, K=K, N=n, block_size=bs)
        ok, err, lim = O.tolerance_ok(y.cpu().numpy(), ref, np.float16)
        assert ok, (err, lim)
    r = (A.astype(np.float32) + (sk.astype(np.float32) if skip else np.float32(0))).astype(np.float16)
    assert np.array_equal(got[3].cpu().numpy(), r)


@pytest.mark.parametrize("M,K,N,Nkv,bs,zp,skip", CASES + WIDE_MLP)
def test_mlp(gpu, M, K, N, Nkv, bs, zp, skip):
    rng = np.random.default_rng(M + K + N + 1)
    A = rng.standard_normal((M, K)).astype(np.float16)
    sk = rng.standard_normal((M, K)).astype(np.float16) if skip else None
    g = rng.uniform(0.5, 1.5, K).astype(np.float16)
    gw, uw = weights(rng, N, K, bs, zp), weights(rng, N, K, bs, zp)
    gb, ub = ((rng.standard_normal(N) * 0.1).astype(np.float16) for _ in range(2))
    y, _ = ops().matmul_nbits_mlp(dev(A), dev(gw[0]), dev(gw[1]), dev(uw[0]), dev(uw[1]), skip=dev(sk),
                                  norm_scale=dev(g), gate_bias=dev(gb), up_bias=dev(ub), block_size=bs,
                                  gate_zero_points=dev(gw[2]), up_zero_points=dev(uw[2]))
    x = A.astype(np.float64) + (sk.astype(np.float64) if skip else 0)
    x = (x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * g.astype(np.float64)).astype(np.float16)
    h = [O.matmul_nbits(x, w[0], w[1], w[2], None, K=K, N=N, block_size=bs, out_dtype=np.float64) + b.astype(np.float64)
         for w, b in ((gw, gb), (uw, ub))]
    ref = h[0] / (1 + np.exp(-h[0])) * h[1]
    ok, err, lim = O.tolerance_ok(y.cpu().numpy(), ref.astype(np.float16), np.float16)
    assert ok, (err, lim)


@pytest.mark.parametrize("M,N", [(70, 64), (333, 5632)])  # narrow, wide
def test_unaligned_output(gpu, M, N):
    """An output two bytes past a 16-byte boundary (the C entry takes any) is written element by element."""
    from xrgpu_amd import _native as nat
    K, bs = 128, 32
    rng = np.random.default_rng(M)
    A = dev(rng.standard_normal((M, K)).astype(np.float16))
    g, u = ([dev(t) for t in weights(rng, N, K, bs, None)[:2]] for _ in range(2))
    gm = dev(rng.uniform(0.5, 1.5, K).astype(np.float16))
    want, _ = ops().matmul_nbits_mlp(A, *g, *u, norm_scale=gm, block_size=bs)
    buf = torch.full((M * N + 16,), 7.0, dtype=torch.float16, device="cuda")
    ws = torch.empty(ops().fused_workspace_bytes("mlp", M, K, N, block_size=bs), dtype=torch.uint8, device="cuda")
    nat.check(nat.lib().xrmm_matmul_nbits_mlp_ws(
        A.data_ptr(), None, gm.data_ptr(), g[0].data_ptr(), g[1].data_ptr(), None, None, u[0].data_ptr(), u[1].data_ptr(),
        None, None, nat.UNSPECIFIED, buf.data_ptr() + 2, None, M, K, N, 4, bs, 1e-5, nat.ACT["silu"], nat.F16, ws.data_ptr(),
        ws.numel(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(buf[1:1 + M * N].view(M, N), want)
    assert (buf[:1] == 7).all() and (buf[1 + M * N:] == 7).all()


def test_two_gib_of_activations(gpu):
    """Activations that end 32 bytes below 2^31: the K groups' step past the last row
    reads zeros, not the first row's infinities."""
    M, K, N, bs = 8191, 131088, 8, 32
    rng = np.random.default_rng(4)
    g, u = ([dev(t) for t in weights(rng, N, K, bs, None)[:2]] for _ in range(2))
    A = torch.zeros((M, K), dtype=torch.float16, device="cuda")
    A[:2] = float("inf")
    A[-70:] = torch.randn(70, K, device="cuda", generator=torch.Generator("cuda").manual_seed(2)).half()
    y, _ = ops().matmul_nbits_mlp(A, *g, *u, block_size=bs)
    want, _ = ops().matmul_nbits_mlp(A[-70:].contiguous(), *g, *u, block_size=bs)
    assert torch.equal(y[-70:], want) and torch.isfinite(want).all()
