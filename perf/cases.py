"""The calls that users of this framework time: the quantised projections, MoE
layers and embedding lookups of a transformer, through ``xrgpu_amd.ops``.

A case names one operator ("op") and its sizes. ``listed()`` holds fixed calls,
``draw()`` makes more over the same ranges: one token to a long prefill, row
counts and widths that are no multiple of any tile, every storage width and
both activation types. Weights are what a model file holds (codes of a rounded
normal distribution, positive block scales), activations are standard normal
as after a normalisation.
"""
import math

import torch

from xrgpu_amd import ops

NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
       -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
       0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)
FP4_MAGNITUDES = (0.0, 0.0052083333333333, 0.6666666666666666, 1.0, 0.3333333333333333, 0.5, 0.1666666666666666, 0.25)


def listed():
    return [
        # one token through an FFN up-projection: the decode step of an 8B model
        dict(name="matmul_decode_m1", op="matmul", dtype="f16", M=1, K=4096, N=14336, bits=4, bs=32, zp="none",
             bias=False),
        # a ragged continuous batch through the FFN down-projection
        dict(name="matmul_batch_m37", op="matmul", dtype="f16", M=37, K=14336, N=4096, bits=4, bs=32, zp="packed",
             bias=False),
        # a long prompt through the up-projection, with zero points and a bias
        dict(name="matmul_prefill_m2048", op="matmul", dtype="f16", M=2048, K=4096, N=14336, bits=4, bs=128,
             zp="packed", bias=True),
        # a float32 graph's prompt (the T1 = float32 form of the contract), ragged rows
        dict(name="matmul_f32_prefill_m509", op="matmul", dtype="f32", M=509, K=2560, N=4096, bits=4, bs=64,
             zp="none", bias=False),
        # normalisation and the three attention projections of a small decode batch (GQA)
        dict(name="qkv_decode_m4", op="qkv", dtype="f16", M=4, K=4096, N=4096, Nkv=1024, bs=64, zp="packed",
             skip=False),
        # gate and up projections of a decode batch
        dict(name="mlp_batch_m16", op="mlp", dtype="f16", M=16, K=4096, N=14336, bs=32, zp="none", skip=False,
             norm=False),
        # residual add, normalisation, gate and up for a ragged prompt of a 1B model
        dict(name="mlp_prefill_m333", op="mlp", dtype="f16", M=333, K=2048, N=5632, bs=32, zp="none", skip=True,
             norm=True),
        # one token through a mixture-of-experts layer (8 experts, 2 taken)
        dict(name="qmoe_decode_t1", op="qmoe", T=1, H=4096, I=14336, E=8, k=2, bits=4, bs=64, act="swiglu"),
        # a prompt through the same layer
        dict(name="qmoe_prefill_t300", op="qmoe", T=300, H=4096, I=14336, E=8, k=2, bits=4, bs=64, act="swiglu"),
        # NF4 weights (the bitsandbytes format) for a prompt
        dict(name="bnb4_prefill_m250", op="bnb4", dtype="f16", M=250, K=4096, N=11008, bs=64, quant=1),
        # accuracy level 4 (int8 activations) for a prompt
        dict(name="int8a_prefill_m384", op="int8a", dtype="f16", M=384, K=4096, N=4096, bs=32, zp="none",
             bias=False),
        # the quantised embedding table: a prompt's rows
        dict(name="gather_embed_n2048", op="gather", rows=128256, width=4096, bits=4, bs=32, zp=False, n=2048),
    ]


# The most multiply-adds a drawn case of an operator has: no more than the
# listed prompt of that operator (matmul: float16 4-bit, others).
_MOST = {"matmul": 2048 * 4096 * 14336, "matmul_other": 509 * 2560 * 4096, "qkv": 333 * 2048 * 5632 * 2,
         "mlp": 333 * 2048 * 5632 * 2, "qmoe": 300 * 2 * 3 * 4096 * 14336, "bnb4": 250 * 4096 * 11008,
         "int8a": 384 * 4096 * 4096}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("matmul", "matmul", "matmul", "qkv", "mlp", "qmoe", "qmoe", "bnb4", "int8a", "gather"))
    bs = rng.choice((32, 32, 64, 128))
    if op == "gather":
        return dict(op=op, rows=_log(rng, 8000, 128256), width=bs * rng.randint(1024 // bs, 5120 // bs),
                    bits=rng.choice((4, 4, 8)), bs=bs, zp=rng.random() < 0.4, n=_log(rng, 16, 2048))
    if op == "qmoe":
        E = rng.choice((8, 16, 32))
        H = 128 * rng.randint(8, 32)
        I = 128 * rng.randint(6, min(112, 112 * 8 // E))
        k, T = rng.choice((1, 2, 2, 4)), _log(rng, 1, 512)
        T = max(1, min(T, _MOST["qmoe"] // (k * 3 * H * I)))
        return dict(op=op, T=T, H=H, I=I, E=E, k=k, bits=rng.choice((4, 4, 4, 8)), bs=rng.choice((0, 32, 64, 128)),
                    act=rng.choice(("swiglu", "swiglu", "relu")))
    N = _log(rng, 512, 14336)
    if rng.random() < 0.6:
        N = (N + 63) // 64 * 64
    unit = 128 if op == "int8a" else bs
    K = unit * max(1024 // unit, _log(rng, 1024, 14336) // unit)
    M = _log(rng, 1, 2048 if op == "matmul" else 512)
    zp = rng.choice(("none", "none", "packed"))
    if op == "matmul":
        dtype, bits = rng.choice((("f16", 4), ("f16", 4), ("f16", 4), ("f32", 4), ("f16", 8), ("f16", 2)))
        if zp == "packed" and rng.random() < 0.3:
            zp = "float"
        if rng.random() < 0.2:
            K -= 8  # a last block that is not whole
        M = max(1, min(M, _MOST["matmul" if (dtype, bits) == ("f16", 4) else "matmul_other"] // (K * N)))
        return dict(op=op, dtype=dtype, M=M, K=K, N=N, bits=bits, bs=bs, zp=zp, bias=rng.random() < 0.3)
    if op == "qkv":
        Nkv = max(64, N // rng.choice((1, 4, 8)))
        M = max(1, min(M, _MOST["qkv"] // (K * (N + 2 * Nkv))))
        return dict(op=op, dtype=rng.choice(("f16", "f16", "f32")), M=M, K=K, N=N, Nkv=Nkv, bs=bs, zp=zp,
                    skip=rng.random() < 0.5)
    if op == "mlp":
        M = max(1, min(M, _MOST["mlp"] // (K * N * 2)))
        return dict(op=op, dtype=rng.choice(("f16", "f16", "f32")), M=M, K=K, N=N, bs=bs, zp=zp,
                    skip=rng.random() < 0.5, norm=rng.random() < 0.7)
    M = max(1, min(M, _MOST[op] // (K * N)))
    if op == "bnb4":
        return dict(op=op, dtype=rng.choice(("f16", "f16", "f32")), M=M, K=K, N=N, bs=bs,
                    quant=rng.choice((1, 1, 1, 0)))
    return dict(op=op, dtype=rng.choice(("f16", "f16", "f32")), M=M, K=K, N=N, bs=bs, zp=zp,
                bias=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# inputs

_DT = {"f16": torch.float16, "f32": torch.float32}


class _Gen:
    def __init__(self, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, device=self.dev, generator=self.g)

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, device=self.dev, generator=self.g) * (hi - lo) + lo

    def randint(self, hi, *shape, dtype=torch.uint8):
        return torch.randint(0, hi, shape, device=self.dev, generator=self.g, dtype=dtype)

    def packed(self, rows, cols, bits):
        """``rows`` x ``cols`` codes of a rounded normal distribution, low-first in bytes."""
        mid, top = 1 << (bits - 1), (1 << bits) - 1
        out = torch.empty((rows, cols * bits // 8), dtype=torch.uint8, device=self.dev)
        step = max(1, (1 << 26) // max(cols, 1))
        for r in range(0, rows, step):
            n = min(step, rows - r)
            c = (self.normal(n, cols) * (mid / 2.8) + mid).round_().clamp_(0, top).to(torch.uint8)
            c = c.view(n, cols * bits // 8, 8 // bits)
            b = c[..., 0].clone()
            for i in range(1, 8 // bits):
                b |= c[..., i] << (bits * i)
            out[r:r + n] = b
        return out

    def scales(self, bits, *shape):
        s = 0.02 * 2.8 / (1 << (bits - 1))  # weights of standard deviation about 0.02
        return self.uniform(0.6 * s, 1.4 * s, *shape)

    def weights(self, N, K, bits, bs, zp, dtype):
        kb = (K + bs - 1) // bs
        w = dict(B=self.packed(N, kb * bs, bits).view(N, kb, bs * bits // 8), S=self.scales(bits, N, kb).to(dtype), Z=None)
        if zp != "none":
            mid = 1 << (bits - 1)
            z = (self.normal(N, kb) + mid).round_().clamp_(0, 2 * mid - 1)
            if zp == "float":
                w["Z"] = (z + 0.25).to(dtype)
            else:
                per = 8 // bits
                z = torch.nn.functional.pad(z.to(torch.uint8), (0, -kb % per)).view(N, -1, per)
                b = z[..., 0].clone()
                for i in range(1, per):
                    b |= z[..., i] << (bits * i)
                w["Z"] = b
        return w


def prepare(case, seed):
    g, c, op = _Gen(seed), case, case["op"]
    if op == "gather":
        blocks = c["width"] // c["bs"]
        return dict(case=c, data=g.packed(c["rows"], c["width"], c["bits"]), scales=g.scales(c["bits"], c["rows"], blocks),
                    zp=g.randint(256, c["rows"], (blocks * c["bits"] + 7) // 8) if c["zp"] else None,
                    idx=g.randint(c["rows"], c["n"], dtype=torch.int32),
                    status=torch.zeros(1, dtype=torch.int32, device=g.dev))
    if op == "qmoe":
        H, I, E, bits, bs = c["H"], c["I"], c["E"], c["bits"], c["bs"]
        F1 = 2 * I if c["act"] == "swiglu" else I
        per = (lambda n: (n // bs,)) if bs else (lambda n: ())
        return dict(case=c, x=g.normal(c["T"], H), router=g.normal(c["T"], E),
                    fc1=g.packed(E * F1, H, bits).view(E, F1, H * bits // 8), s1=g.scales(bits, E, F1, *per(H)),
                    fc2=g.packed(E * H, I, bits).view(E, H, I * bits // 8), s2=g.scales(bits, E, H, *per(I)))
    dtype, M, K, N, bs = _DT[c["dtype"]], c["M"], c["K"], c["N"], c["bs"]
    s = dict(case=c, A=g.normal(M, K).to(dtype))
    if op == "bnb4":  # codes of normal weights fall on the 16 levels about evenly
        s.update(B=g.randint(256, N * K // 2), absmax=g.uniform(0.03, 0.08, N * K // bs).to(dtype))
        return s
    if op in ("matmul", "int8a"):
        s.update(g.weights(N, K, c.get("bits", 4), bs, c["zp"], dtype),
                 bias=(g.normal(N) * 0.1).to(dtype) if c["bias"] else None)
        return s
    s.update(skip=g.normal(M, K).to(dtype) if c["skip"] else None,
             gamma=g.uniform(0.5, 1.5, K).to(dtype) if c.get("norm", True) else None)
    for p, n in (("q", N), ("k", c["Nkv"]), ("v", c["Nkv"])) if op == "qkv" else (("gate", N), ("up", N)):
        s[p] = g.weights(n, K, 4, bs, c["zp"], dtype)
    return s


# ---------------------------------------------------------------------------
# one call

def run(s):
    c, op = s["case"], s["case"]["op"]
    if op == "matmul":
        return ops.matmul_nbits(s["A"], s["B"], s["S"], s["Z"], s["bias"], bits=c["bits"], block_size=c["bs"])
    if op == "qkv":
        q, k, v = s["q"], s["k"], s["v"]
        return ops.matmul_nbits_qkv(s["A"], q["B"], q["S"], k["B"], k["S"], v["B"], v["S"], norm_scale=s["gamma"],
                                    skip=s["skip"], block_size=c["bs"], q_zero_points=q["Z"], k_zero_points=k["Z"],
                                    v_zero_points=v["Z"])
    if op == "mlp":
        g, u = s["gate"], s["up"]
        return ops.matmul_nbits_mlp(s["A"], g["B"], g["S"], u["B"], u["S"], skip=s["skip"], norm_scale=s["gamma"],
                                    block_size=c["bs"], gate_zero_points=g["Z"], up_zero_points=u["Z"],
                                    want_residual=c["skip"])
    if op == "qmoe":
        return ops.qmoe(s["x"], s["router"], s["fc1"], s["s1"], s["fc2"], s["s2"], k=c["k"], activation=c["act"],
                        swiglu_fusion=1 if c["act"] == "swiglu" else 0, expert_weight_bits=c["bits"],
                        block_size=c["bs"])
    if op == "bnb4":
        return ops.matmul_bnb4(s["A"], s["B"], s["absmax"], K=c["K"], N=c["N"], block_size=c["bs"],
                               quant_type=c["quant"])
    if op == "int8a":
        return ops.matmul_nbits_int8a(s["A"], s["B"], s["S"], s["Z"], s["bias"], K=c["K"], N=c["N"],
                                      block_size=c["bs"])
    return ops.gather_block_quantized(s["data"], s["idx"], s["scales"], s["zp"], bits=c["bits"], block_size=c["bs"],
                                      status=s["status"], check=False)


def _weight_bytes(N, K, bits, bs, zp, item):
    kb = (K + bs - 1) // bs
    z = 0 if zp == "none" else kb * item if zp == "float" else (kb * bits + 7) // 8
    return N * (kb * bs * bits // 8 + kb * item + z)


def work(case):
    c, op = case, case["op"]
    if op == "gather":
        blocks = c["width"] // c["bs"]
        row = c["width"] * c["bits"] // 8 + blocks * 4 + ((blocks * c["bits"] + 7) // 8 if c["zp"] else 0)
        return {"bytes": c["n"] * (row + 4 + c["width"] * 4), "flops": c["n"] * c["width"] * 2}
    if op == "qmoe":
        T, H, I, k = c["T"], c["H"], c["I"], c["k"]
        F1 = 2 * I if c["act"] == "swiglu" else I
        # experts that T tokens of k choices each are expected to touch
        used = c["E"] * (1 - (1 - k / c["E"]) ** T)
        n1, n2 = (H // c["bs"], I // c["bs"]) if c["bs"] else (1, 1)
        expert = F1 * (H * c["bits"] // 8 + n1 * 4) + H * (I * c["bits"] // 8 + n2 * 4)
        return {"bytes": used * expert + T * (2 * H + c["E"]) * 4, "flops": 2 * T * k * H * (F1 + I)}
    item, M, K, N, bs = (2 if c["dtype"] == "f16" else 4), c["M"], c["K"], c["N"], c["bs"]
    if op == "bnb4":
        return {"bytes": N * K // 2 + N * K // bs * item + M * (K + N) * item, "flops": 2 * M * K * N}
    if op in ("matmul", "int8a"):
        return {"bytes": _weight_bytes(N, K, c.get("bits", 4), bs, c["zp"], item) + M * (K + N) * item
                + (N * item if c["bias"] else 0), "flops": 2 * M * K * N}
    if op == "qkv":  # the residual comes back in any case
        n, cols, extra = N + 2 * c["Nkv"], N + 2 * c["Nkv"], 2 + (1 if c["skip"] else 0)
    else:
        n, cols, extra = 2 * N, N, 1 + (2 if c["skip"] else 0)
    return {"bytes": _weight_bytes(n, K, 4, bs, c["zp"], item) + M * (cols + extra * K) * item + K * item,
            "flops": 2 * M * K * n}


def tolerance(case):
    if case["op"] == "gather":
        return "exact"  # (code - zero point) * scale, rounded once
    # four times the error against 64 bits: 2.1e-4 .. 3e-4 for binary16 results
    # (4.4e-4 where two projections multiply), 1.2e-7 .. 3.1e-7 for float32 ones
    if case.get("dtype") == "f16":
        return {"rel": 1.8e-3, "max": 1.2e-2} if case["op"] == "mlp" else {"rel": 1.2e-3, "max": 8e-3}
    return {"rel": 1.2e-6, "max": 1.2e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits

def _unpack(B, bits):
    """uint8 [..., n] -> codes [..., n * 8 / bits], low-first."""
    parts = [(B >> (bits * i)) & ((1 << bits) - 1) for i in range(8 // bits)]
    return torch.stack(parts, -1).flatten(-2)


def _dense(w, K, bits, bs):
    """W [N, K] in 64 bits."""
    N, kb = w["S"].shape
    c = _unpack(w["B"].view(N, -1), bits).view(N, kb, bs).double()
    if w["Z"] is None:
        z = torch.full((N, kb), float(1 << (bits - 1)), device=c.device, dtype=torch.float64)
    elif w["Z"].dtype == torch.uint8:
        z = _unpack(w["Z"], bits)[:, :kb].double()
    else:
        z = w["Z"].double()
    return ((c - z[..., None]) * w["S"].double()[..., None]).view(N, kb * bs)[:, :K]


def exact(case, seed):
    s, c, op = prepare(case, seed), case, case["op"]
    if op == "gather":
        rows = s["idx"].long()
        w = dict(B=s["data"][rows], S=s["scales"][rows], Z=None if s["zp"] is None else s["zp"][rows])
        return _dense(w, c["width"], c["bits"], c["bs"])
    if op == "qmoe":
        T, H, E, k, bits = c["T"], c["H"], c["E"], c["k"], c["bits"]
        x, top = s["x"].double(), s["router"].double().topk(k, dim=1)
        weight = torch.zeros(T, E, dtype=torch.float64, device=x.device).scatter_(1, top.indices, top.values.softmax(1))
        y = torch.zeros(T, H, dtype=torch.float64, device=x.device)

        def expert(codes, scales, e, cols):
            q = _unpack(codes[e], bits).double() - (1 << (bits - 1))
            sc = scales[e].double()
            return q * (sc[:, None] if sc.dim() == 1 else sc.repeat_interleave(c["bs"], 1))[:, :cols]

        for e in range(E):
            t = weight[:, e].nonzero()[:, 0]
            if not len(t):
                continue
            h = x[t] @ expert(s["fc1"], s["s1"], e, H).T
            h = torch.nn.functional.silu(h[:, 0::2]) * h[:, 1::2] if c["act"] == "swiglu" else h.relu()
            y[t] += weight[t, e][:, None] * (h @ expert(s["fc2"], s["s2"], e, c["I"]).T)
        return y
    M, K, N, bs = c["M"], c["K"], c["N"], c["bs"]
    A = s["A"].double()
    if op == "bnb4":
        book = NF4 if c["quant"] == 1 else FP4_MAGNITUDES + tuple(-v for v in FP4_MAGNITUDES)
        q = torch.stack((s["B"] >> 4, s["B"] & 15), -1).view(N, K // bs, bs)  # high nibble first
        W = torch.tensor(book, dtype=torch.float64, device=A.device)[q.int()]
        return A @ (W * s["absmax"].double().view(N, K // bs, 1)).view(N, K).T
    if op in ("matmul", "int8a"):
        if op == "int8a":  # rows rounded to 8 bits per 128 values, scale and quotient in 32 bits
            b = s["A"].float().view(M, K // 128, 128)
            step = (b.abs().amax(2, keepdim=True).double() / 127).float()
            A = ((b.double() / step.double()).float().round().clamp(-127, 127).double() * step.double()).view(M, K)
        y = A @ _dense(s, K, c.get("bits", 4), bs).T
        return y if s["bias"] is None else y + s["bias"].double()
    r = A if s["skip"] is None else A + s["skip"].double()
    x = r
    if s["gamma"] is not None:
        eps = 1e-6 if op == "qkv" else 1e-5
        x = r / (r.square().mean(1, keepdim=True) + eps).sqrt() * s["gamma"].double()
    if op == "qkv":
        return tuple(x @ _dense(s[p], K, 4, bs).T for p in ("q", "k", "v")) + (r,)
    gate, up = (x @ _dense(s[p], K, 4, bs).T for p in ("gate", "up"))
    return torch.nn.functional.silu(gate) * up, (r if c["skip"] else None)
