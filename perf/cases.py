"""Performance cases of the framework's public entry points on one GPU.

Every case is a plain dict; ``prepare`` makes what a user's program holds
before the call (inputs, weights), ``run`` is one pass through the public API,
``exact`` is the same result in 64-bit plain torch.  Kinds:

* ``ring``: :func:`harp_amd.ring_attention`, one rank's share of the ring on
  one GPU, forward only (``infer``) or forward + backward (``train``);
* ``qk``: the step before it, RMSNorm and / or RoPE of one of q, k;
* ``project``: the producer, :func:`harp_amd.project_qkv`;
* ``block``: :class:`harp_amd.RingZAttention`, the whole attention block;
* ``linear``: :func:`harp_amd.xhblas_gemm`, a Linear layer's product.
"""

from __future__ import annotations

import math

import torch
from torch import nn

import harp_amd
from harp_amd.gemm import NO_TRANS, REFERENCE_SHAPES, ROW_MAJOR

DEV = "cuda:0"
EPS = 1e-5


def _ring(name, B, H, D, T, sp, valid=None, chunk=None, rank=0, mode="train"):
    """T query rows against sp chunks of ``chunk`` stored rows, the first
    ``valid`` of them unmasked."""
    chunk = T if chunk is None else chunk
    case = {"kind": "ring", "B": B, "H": H, "D": D, "T": T, "sp": sp, "chunk": chunk,
            "valid": chunk if valid is None else valid, "rank": rank, "mode": mode}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one small attention layer in training: latency and launches
        _ring("ring_single", 1, 8, 64, 512, 1),
        # the model's own per-rank call in training: 30 heads, 256 or 768
        # local tokens, 8 ranks' chunks
        _ring("ring_rank256", 1, 30, 128, 256, 8),
        _ring("ring_rank768", 1, 30, 128, 768, 8),
        # a 1024-token image sampled on one GPU: forward only, one chunk
        _ring("ring_infer1024", 1, 30, 128, 1024, 1, mode="infer"),
        # training at the narrower head dims
        _ring("ring_d64", 1, 16, 64, 2048, 4),
        _ring("ring_d72", 2, 16, 72, 4096, 8),
        # 4096 image + 333 text tokens, chunks padded to 4480 rows and masked
        _ring("ring_ragged", 1, 24, 128, 4429, 4, valid=4429, chunk=4480),
        # long-context training, the largest call
        _ring("ring_long", 1, 24, 128, 8192, 8),
        # RMSNorm + RoPE of q (or k) as separate operators, forward + backward
        {"name": "qk_train", "kind": "qk", "op": "norm_rope", "B": 1, "H": 24, "D": 128, "S": 8192},
        # the q/k/v producer in training
        {"name": "project_train", "kind": "project", "B": 1, "H": 24, "S": 8192, "mode": "train"},
        # the whole attention block in training at the model width, 256 tokens a rank
        {"name": "block_train", "kind": "block", "B": 1, "H": 30, "S": 2048, "sp": 8, "mode": "train"},
        # a feed-forward Linear of 768 tokens
        {"name": "linear_ffn", "kind": "linear", "M": 768, "N": 10240, "K": 3840, "ta": 111, "tb": 112},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ring"] * 6 + ["qk"] * 2 + ["project", "block", "linear"])
    mode = rng.choice(["train", "train", "infer"])
    if kind == "ring":
        while True:
            D = rng.choice([64, 72, 128, 128])
            B, H, sp = rng.choice([1, 1, 2]), rng.choice([8, 16, 24, 30]), rng.choice([1, 1, 2, 4, 8])
            T = _log_int(rng, 64, 8192)
            pad = rng.choice([0, 0, rng.randint(1, 128)])
            case = _ring(None, B, H, D, T, sp, valid=T, chunk=T + pad, rank=rng.randrange(sp), mode=mode)
            if work(case)["flops"] <= 2.3e13:
                return case
    if kind == "qk":
        return {"kind": "qk", "op": rng.choice(["norm_rope", "norm_rope", "norm", "rope"]), "B": rng.choice([1, 2]),
                "H": rng.choice([8, 16, 24, 30]), "D": rng.choice([64, 72, 128]), "S": _log_int(rng, 256, 16384)}
    if kind == "project":
        return {"kind": "project", "B": 1, "H": rng.choice([24, 30]), "S": _log_int(rng, 256, 8192), "mode": mode}
    if kind == "block":
        sp = rng.choice([1, 2, 4, 8])
        return {"kind": "block", "B": 1, "H": rng.choice([24, 30]), "S": sp * _log_int(rng, 512 // sp, 4608 // sp),
                "sp": sp, "mode": mode}
    M, N, K, ta, tb = rng.choice([s for g in ("demo1", "demo2", "vector") for s in REFERENCE_SHAPES[g]])
    return {"kind": "linear", "M": M, "N": N, "K": K, "ta": ta, "tb": tb}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Norm(nn.Module):
    def __init__(self, d):
        super().__init__()
        self.eps = EPS
        self.weight = nn.Parameter(torch.ones(d, dtype=torch.bfloat16, device=DEV))


class _Attention(nn.Module):
    """The attributes RingZAttention and project_qkv read of the model's attention module."""

    def __init__(self, dim, heads, d):
        super().__init__()

        def linear(n_in, n_out):
            return nn.Linear(n_in, n_out, bias=False, dtype=torch.bfloat16, device=DEV)

        self.heads = heads
        self.to_q, self.to_k, self.to_v = linear(dim, heads * d), linear(dim, heads * d), linear(dim, heads * d)
        self.norm_q, self.norm_k = _Norm(d), _Norm(d)
        self.to_out = nn.ModuleList([linear(heads * d, dim), nn.Identity()])


def _normal(g, *shape, scale=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, device=DEV, generator=g) * scale).to(dtype)


def _heads(g, B, H, T, D, scale=1.0):
    """[B, H, T, D] view of token-major [B, T, H, D] storage, as the model's projections give it."""
    return _normal(g, B, T, H, D, scale=scale).transpose(1, 2)


def _freqs(S, D):
    """The RoPE table: exp(i * position * theta^(-2p/D)), complex64 [S, D/2]."""
    inv = 256.0 ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    ang = torch.arange(S, dtype=torch.float64)[:, None] * inv[None, :]
    return torch.polar(torch.ones_like(ang), ang).to(torch.complex64).to(DEV)


def _module(g, H):
    dim = H * 128
    m = _Attention(dim, H, 128)
    with torch.no_grad():
        for lin in (m.to_q, m.to_k, m.to_v, m.to_out[0]):
            lin.weight.copy_(_normal(g, dim, dim, scale=dim ** -0.5))
        for nm in (m.norm_q, m.norm_k):
            nm.weight.copy_(1.0 + _normal(g, 128, scale=0.1, dtype=torch.float32))
    return m


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 3407)
    train = case.get("mode", "train") == "train"
    st = {"case": case}
    if case["kind"] == "ring":
        B, H, D, T, L = case["B"], case["H"], case["D"], case["T"], case["sp"] * case["chunk"]
        scale = 0.5 if D == 72 else 1.0
        st["q"], st["k"], st["v"] = (_heads(g, B, H, n, D, scale).requires_grad_(train) for n in (T, L, L))
        st["dout"] = _heads(g, B, H, T, D, scale) if train else None
        st["lens"] = [case["valid"]] * case["sp"] if case["valid"] != case["chunk"] else None
    elif case["kind"] == "qk":
        B, H, D, S = case["B"], case["H"], case["D"], case["S"]
        st["x"] = _heads(g, B, H, S, D).requires_grad_(True)
        st["dy"] = _heads(g, B, H, S, D)
        st["w"] = (1.0 + _normal(g, D, scale=0.1, dtype=torch.float32)).to(torch.bfloat16).requires_grad_(True)
        st["freqs"] = _freqs(S, D)
    elif case["kind"] in ("project", "block"):
        B, H, S = case["B"], case["H"], case["S"]
        st["m"] = _module(g, H).requires_grad_(train)
        st["x"] = _normal(g, B, S, H * 128).requires_grad_(train)
        st["freqs"] = _freqs(S, 128)
        if case["kind"] == "block":
            st["layer"] = harp_amd.RingZAttention(st["m"], case["sp"])
            st["dout"] = _normal(g, B, S, H * 128)
        else:
            st["dout"] = tuple(_heads(g, B, H, S, 128) for _ in range(3))
    else:
        M, N, K = case["M"], case["N"], case["K"]
        st["A"] = _normal(g, *((M, K) if case["ta"] == NO_TRANS else (K, M)))
        st["W"] = _normal(g, *((K, N) if case["tb"] == NO_TRANS else (N, K)), scale=K ** -0.5)
        st["C"] = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    return st


def _params(st):
    m = st["m"]
    ws = [st["x"], m.to_q.weight, m.to_k.weight, m.to_v.weight, m.norm_q.weight, m.norm_k.weight]
    return ws + [m.to_out[0].weight] if st["case"]["kind"] == "block" else ws


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    train = case.get("mode", "train") == "train"
    if kind == "linear":
        M, N, K, A, W = case["M"], case["N"], case["K"], st["A"], st["W"]
        rc = harp_amd.xhblas_gemm(ROW_MAJOR, case["ta"], case["tb"], M, N, K, 1.0, A, A.size(1), W, W.size(1), 0.0,
                                  st["C"], N)
        if rc != 0:
            raise RuntimeError(f"xhblas_gemm returned {rc}")
        return st["C"]
    if kind == "qk":
        x, w, f = st["x"], st["w"], st["freqs"]
        if case["op"] == "norm_rope":
            y = harp_amd.QKNormRopeFn.apply(x, w, f, EPS)
        elif case["op"] == "norm":
            y = harp_amd.RMSNormFn.apply(x, w, EPS)
        else:
            y = harp_amd.ApplyRotaryComplexFn.apply(x, f)
        return (y, *torch.autograd.grad(y, (x,) if case["op"] == "rope" else (x, w), st["dy"]))
    with torch.set_grad_enabled(train):
        if kind == "ring":
            y = harp_amd.ring_attention(st["q"], st["k"], st["v"], case["sp"], case["rank"], st["lens"])
            wrt = (st["q"], st["k"], st["v"])
        elif kind == "project":
            y = harp_amd.project_qkv(st["m"], st["x"], st["freqs"])
            wrt = _params(st)
        else:
            y = st["layer"](st["x"], st["freqs"])
            wrt = _params(st)
    outs = y if isinstance(y, tuple) else (y,)
    if not train:
        return outs
    return (*outs, *torch.autograd.grad(outs, wrt, st["dout"] if isinstance(st["dout"], tuple) else (st["dout"],)))


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------

def work(case):
    train = case.get("mode", "train") == "train"
    if case["kind"] == "ring":
        rows_q, rows_k = case["B"] * case["H"] * case["T"], case["B"] * case["H"] * case["sp"] * case["valid"]
        # q, k, v in and o out; in training dO in, dq, dk, dv out
        el = (4 * rows_q + 4 * rows_k if train else 2 * rows_q + 2 * rows_k) * case["D"]
        return {"bytes": 2 * el, "flops": (14 if train else 4) * rows_q * case["sp"] * case["valid"] * case["D"]}
    if case["kind"] == "qk":
        n = case["B"] * case["H"] * case["S"] * case["D"]
        table = (0 if case["op"] == "norm" else 4) * case["S"] * case["D"]
        # x in, y out, dy in, dx out
        return {"bytes": 8 * n + table, "flops": (10 if case["op"] == "rope" else 30) * n}
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    M, dim = case["B"] * case["S"], case["H"] * 128
    n_lin = 3 if case["kind"] == "project" else 4
    flops = 2 * M * dim * dim * n_lin * (3 if train else 1)
    if case["kind"] == "block":
        flops += (14 if train else 4) * case["B"] * case["S"] * case["S"] * dim
        el = (2 + n_lin * dim / M) * M * dim * (2 if train else 1)
    else:
        el = (1 + 3 + 3 * dim / M) * M * dim * (2 if train else 1)
    return {"bytes": int(2 * el), "flops": flops}


def tolerance(case):
    if case["kind"] in ("qk", "linear"):
        # fp32 arithmetic and one bf16 result per stage: another order of the
        # sums moves single results by one bf16 unit (1e-5 to 5e-5 measured,
        # 4e-4 for one unit in a 128-element weight gradient)
        return {"rel": 1e-3}
    # outputs are bf16 and so are the probabilities (and, in training, dS and
    # the producer's results) as matrix operands: 3.5e-3 measured between
    # other orders of the sums, other chunkings and the unfused producer
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _attention64(q, k, v, dout=None):
    """softmax(q k^T / sqrt(D)) v of [B, H, T, D], and its gradients for dout, in row blocks."""
    q, k, v = q.detach().double(), k.detach().double(), v.detach().double()
    scale = 1.0 / math.sqrt(q.size(-1))
    o = torch.empty_like(q)
    grads = None if dout is None else (torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v))
    rows = max(64, min(q.size(2), (1 << 28) // k.size(2)))
    for b in range(q.size(0)):
        for h in range(q.size(1)):
            kk, vv = k[b, h].contiguous(), v[b, h].contiguous()
            for r in range(0, q.size(2), rows):
                qq = q[b, h, r:r + rows].contiguous()
                p = torch.softmax((qq @ kk.t()) * scale, dim=-1)
                o[b, h, r:r + rows] = p @ vv
                if dout is None:
                    continue
                dd = dout[b, h, r:r + rows].double().contiguous()
                dv = p.t() @ dd
                ds = dd @ vv.t()
                ds -= (dd * o[b, h, r:r + rows]).sum(-1, keepdim=True)
                ds *= p
                ds *= scale
                grads[0][b, h, r:r + rows] = ds @ kk
                grads[1][b, h] += ds.t() @ qq
                grads[2][b, h] += dv
    return o, grads


class _Attention64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v):
        ctx.save_for_backward(q, k, v)
        return _attention64(q, k, v)[0]

    @staticmethod
    def backward(ctx, dout):
        return _attention64(*ctx.saved_tensors, dout)[1]


def _norm64(x, w):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _rope64(x, freqs):
    c = torch.view_as_complex(x.reshape(*x.shape[:-1], -1, 2).contiguous()) * freqs.to(torch.complex128)
    return torch.view_as_real(c).flatten(-2)


def exact(case, seed):
    st = prepare(case, seed)
    train = case.get("mode", "train") == "train"
    if case["kind"] == "ring":
        keep = torch.arange(case["sp"] * case["chunk"], device=DEV) % case["chunk"] < case["valid"]
        o, grads = _attention64(st["q"], st["k"][:, :, keep], st["v"][:, :, keep], st["dout"])
        if not train:
            return (o,)
        out = [o, grads[0]]
        for g in grads[1:]:
            full = torch.zeros_like(st["k"], dtype=torch.float64)
            full[:, :, keep] = g
            out.append(full)
        return tuple(out)
    if case["kind"] == "linear":
        a, w = st["A"].double(), st["W"].double()
        return (a if case["ta"] == NO_TRANS else a.t()) @ (w if case["tb"] == NO_TRANS else w.t())
    if case["kind"] == "qk":
        x, w = st["x"].detach().double().requires_grad_(True), st["w"].detach().double().requires_grad_(True)
        y = x if case["op"] == "rope" else _norm64(x, w)
        y = y if case["op"] == "norm" else _rope64(y, st["freqs"])
        return (y.detach(), *torch.autograd.grad(y, (x,) if case["op"] == "rope" else (x, w), st["dy"].double()))
    p = [t.detach().double().requires_grad_(train) for t in _params(st)]
    x = p[0]

    def split(t):
        return t.view(x.size(0), x.size(1), case["H"], 128).transpose(1, 2)

    q, k, v = (split(x @ w.t()) for w in p[1:4])
    q, k = _rope64(_norm64(q, p[4]), st["freqs"]), _rope64(_norm64(k, p[5]), st["freqs"])
    if case["kind"] == "project":
        outs, douts = (q, k, v), st["dout"]
    else:
        outs, douts = (_Attention64.apply(q, k, v).transpose(1, 2).flatten(2, 3) @ p[6].t(),), (st["dout"],)
    res = tuple(t.detach() for t in outs)
    if not train:
        return res
    return (*res, *torch.autograd.grad(outs, p, tuple(d.double() for d in douts)))
