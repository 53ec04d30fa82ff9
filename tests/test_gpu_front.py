"""GPU: the native front end of ops.py takes ordinary calls, gives what the Python
checks' path gives, and leaves everything else to them: other layouts, dtypes and
devices, tensor subclasses, functorch and dispatch modes, empty batches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture
def both(gpu):
    """run(f): f() with the native front end and without it, equal results."""
    from xrgpu_amd import ops
    assert ops._front(), "the native front end is not built"

    def run(f):
        front = ops._FRONT
        a = f()
        ops._FRONT = False
        try:
            b = f()
        finally:
            ops._FRONT = front
        for x, y in zip(a if isinstance(a, tuple) else (a,), b if isinstance(b, tuple) else (b,)):
            assert (x is None) == (y is None)
            if x is not None:
                assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)
        return a
    return run


def q(g, N, K, bs, bits, zp, dt):
    kb = -(-K // bs)
    B = torch.randint(0, 256, (N, kb, bs * bits // 8), dtype=torch.uint8, device="cuda", generator=g)
    S = (torch.rand(N, kb, device="cuda", generator=g) * 0.02).to(dt)
    Z = None
    if zp == "packed":
        Z = torch.randint(0, 256, (N, (kb * bits + 7) // 8), dtype=torch.uint8, device="cuda", generator=g)
    elif zp is not None:
        Z = (torch.rand(N, kb, device="cuda", generator=g) * 8 + 4).to(zp)
    return B, S, Z


@pytest.mark.parametrize("lead,K,N,bs,bits,zp,dt", [
    ((1,), 128, 40, 32, 4, None, torch.float16), ((2, 2), 96, 33, 32, 4, "packed", torch.float16),
    ((3,), 200, 17, 64, 8, torch.float32, torch.float32), ((70,), 256, 64, 64, 2, "packed", torch.float16),
    ((4,), 128, 24, 16, 4, torch.float16, torch.float16)])
def test_matmul(both, lead, K, N, bs, bits, zp, dt):
    from xrgpu_amd import ops
    g = torch.Generator("cuda").manual_seed(K + N)
    A = torch.randn(*lead, K, device="cuda", generator=g).to(dt)
    B, S, Z = q(g, N, K, bs, bits, zp, dt)
    bias = torch.randn(N, device="cuda", generator=g).to(dt)
    y = both(lambda: ops.matmul_nbits(A, B, S, Z, bias, bits=bits, block_size=bs))
    assert y.shape == (*lead, N)


@pytest.mark.parametrize("M,dt,zp,skip,res", [(4, torch.float16, "packed", False, True), (1, torch.float32, None, True, False),
                                              (80, torch.float16, None, True, True)])
def test_qkv_mlp(both, M, dt, zp, skip, res):
    from xrgpu_amd import ops
    K, N, Nkv, bs = 256, 96, 40, 64
    g = torch.Generator("cuda").manual_seed(M)
    A = torch.randn(M, K, device="cuda", generator=g).to(dt)
    sk = torch.randn(M, K, device="cuda", generator=g).to(dt) if skip else None
    gm = torch.rand(K, device="cuda", generator=g).to(dt)
    a, b, c = (q(g, n, K, bs, 4, zp, dt) for n in (N, Nkv, Nkv))
    both(lambda: ops.matmul_nbits_qkv(A, a[0], a[1], b[0], b[1], c[0], c[1], norm_scale=gm, skip=sk, block_size=bs,
                                      q_zero_points=a[2], k_zero_points=b[2], v_zero_points=c[2], want_residual=res))
    both(lambda: ops.matmul_nbits_qkv(A, a[0], a[1], b[0], b[1], c[0], c[1], norm_scale=gm, block_size=bs, epsilon=1,
                                      q_zero_points=a[2], k_zero_points=b[2], v_zero_points=c[2]))
    u = q(g, N, K, bs, 4, zp, dt)
    both(lambda: ops.matmul_nbits_mlp(A, a[0], a[1], u[0], u[1], skip=sk, norm_scale=gm if skip else None, block_size=bs,
                                      activation="gelu", gate_zero_points=a[2], up_zero_points=u[2], want_residual=res))


@pytest.mark.parametrize("M,K,N,bits,dt", [(17, 512, 256, 4, torch.float32), (20, 256, 96, 8, torch.float16),
                                           (128, 2048, 256, 4, torch.float16)])
def test_workspace_call(both, M, K, N, bits, dt):
    """A call that runs on a workspace comes back from the front end checked, as its bytes."""
    from xrgpu_amd import ops
    g = torch.Generator("cuda").manual_seed(M)
    A = torch.randn(M, K, device="cuda", generator=g).to(dt)
    B, S, Z = q(g, N, K, 32, bits, "packed", dt)
    need = ops.matmul_nbits_workspace_bytes(M, K, N, bits, 32, dt)
    assert need > 0 and ops._front().matmul(A, B, S, Z, None, None, None, bits, 32) == need
    assert ops._front().matmul(A, B, S, Z[:, :-1], None, None, None, bits, 32) is None
    both(lambda: ops.matmul_nbits(A, B, S, Z, bits=bits))


def test_streams_and_threads(gpu):
    """Each thread's calls run on its own stream, after the work enqueued there."""
    from concurrent.futures import ThreadPoolExecutor
    from xrgpu_amd import ops
    g = torch.Generator("cuda").manual_seed(4)
    B, S, Z = q(g, 96, 512, 32, 4, "packed", torch.float16)
    As = [torch.randn(m, 512, device="cuda", generator=g).half() for m in (2, 70, 3, 130)]
    want = [ops.matmul_nbits(2 * a, B, S, Z) for a in As]
    torch.cuda.synchronize()

    def work(a):
        with torch.cuda.stream(torch.cuda.Stream()):
            ys = []
            for _ in range(8):
                x = torch.zeros_like(a)
                for _ in range(2):
                    x += a
                ys.append(ops.matmul_nbits(x, B, S, Z))
            torch.cuda.current_stream().synchronize()
            return ys

    with ThreadPoolExecutor(4) as pool:
        for ys, w in zip(pool.map(work, As), want):
            assert all(torch.equal(y, w) for y in ys)


def test_bnb4_gather(both):
    from xrgpu_amd import ops
    g = torch.Generator("cuda").manual_seed(3)
    A = torch.randn(3, 128, device="cuda", generator=g).half()
    B = torch.randint(0, 256, (40 * 64,), dtype=torch.uint8, device="cuda", generator=g)
    am = torch.rand(40 * 2, device="cuda", generator=g).half()
    both(lambda: ops.matmul_bnb4(A, B, am, K=128, N=40, block_size=64))
    D = torch.randint(0, 256, (50, 64), dtype=torch.uint8, device="cuda", generator=g)
    S = torch.rand(50, 4, device="cuda", generator=g)
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    for dt in (torch.int32, torch.int64):
        idx = torch.tensor([3, 49, 0], dtype=dt, device="cuda")
        both(lambda: ops.gather_block_quantized(D, idx, S, bits=4, block_size=32, status=st, check=False))
        both(lambda: ops.gather_block_quantized(D, idx, S, bits=4, block_size=32, status=st.view(torch.uint32), check=False))


def test_declines(gpu):
    """What the front end does not take raises or runs as the Python path does."""
    from torch.utils._python_dispatch import TorchDispatchMode
    from xrgpu_amd import _native as nat, ops
    front = ops._front()
    g = torch.Generator("cuda").manual_seed(5)
    A = torch.randn(2, 128, device="cuda", generator=g).half()
    B, S, Z = q(g, 40, 128, 32, 4, None, torch.float16)

    def native(a=A, b=B, s=S, z=None, bias=None, K=None, N=None, bits=4, bs=32):
        return front.matmul(a, b, s, z, bias, K, N, bits, bs)
    assert native() is not None

    class Sub(torch.Tensor):
        pass

    wide = torch.randn(2, 256, device="cuda").half()
    for kw in (dict(a=wide[:, :128]), dict(a=A.cpu()), dict(a=A.double()), dict(a=A[:0]), dict(s=S.float()), dict(b=B[:39]),
               dict(b=B.view(torch.int8)), dict(K=96), dict(N=39), dict(bits=3), dict(bs=64), dict(a=A.as_subclass(Sub)),
               dict(bias=S[0]), dict(z=Z if Z is not None else S[:, :1]), dict(bits=4.0), dict(a=None)):
        assert native(**kw) is None, kw
    with pytest.raises(nat.XrmmInvalid, match="contiguous"):
        ops.matmul_nbits(wide[:, :128], B, S, block_size=32)
    with pytest.raises(nat.XrmmInvalid, match="scales"):
        ops.matmul_nbits(A, B, S.float(), block_size=32)
    assert ops.matmul_nbits(A[:0], B, S, block_size=32).shape == (0, 40)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert native() is None
    seen = []
    torch.func.vmap(lambda a: seen.append(native(a=a)) or a)(A[None])
    assert seen == [None]


def test_error_through_front(gpu):
    """A call the library refuses raises through the front end."""
    from xrgpu_amd import _native as nat, ops
    D = torch.zeros((4, 6), dtype=torch.uint8, device="cuda")
    S = torch.ones((4, 2), device="cuda")
    idx = torch.zeros(2, dtype=torch.int32, device="cuda")
    st = torch.zeros(1, dtype=torch.int32, device="cuda")
    front = ops._front()
    errs = []
    for f in (front, False):
        ops._FRONT = f
        try:
            ops.gather_block_quantized(D, idx, S, bits=4, block_size=8, status=st, check=False)
            errs.append(None)
        except (nat.XrmmInvalid, nat.XrmmError) as e:
            errs.append((type(e), str(e)))
        finally:
            ops._FRONT = front
    assert errs[0] == errs[1]


def test_graph_replay(gpu):
    """Captured through the front end, replayed with eager work between: every replay right."""
    from xrgpu_amd import ops
    g = torch.Generator("cuda").manual_seed(9)
    A = torch.randn(2, 256, device="cuda", generator=g).half()
    B, S, _ = q(g, 96, 256, 32, 4, None, torch.float16)
    ops.matmul_nbits(A, B, S, block_size=32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ops.matmul_nbits(A, B, S, block_size=32)
    for i in range(4):
        A.copy_(torch.randn(2, 256, device="cuda", generator=g).half())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.matmul_nbits(A, B, S, block_size=32))
