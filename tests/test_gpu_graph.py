"""HIP-graph capture of the block's operators: ring-attention forward, delta
and backward and the one-call attend and grad (torch.ops.ring_attention_ops),
with whole grids and with split ones (partials and merges in the graph), the
fused QK RMSNorm + RoPE
forward and backward (torch.ops.async_op) and the fused q/k/v projection
kernel (harp_amd.qkv) are recorded once into a
torch.cuda.CUDAGraph on static tensors and replayed on new inputs.  No
operator allocates device memory outside torch's allocator or clears memory
with hipMemsetAsync, so each replay must equal the eager result on the same
inputs bit for bit.  Between replays the test runs its own eager work and
synchronizes, and it checks every replay."""

import math

import pytest
import torch

import harp_amd
from harp_amd import _lib
from tests.gpu_harness import split_plan

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _inputs(seed, B=1, H=2, T=256, D=64, N=2):
    g = torch.Generator().manual_seed(seed)

    def tok(t):  # token-major storage seen as [B, H, T, D]
        return (torch.randn((B, t, H, D), generator=g)).to(torch.bfloat16).to(DEV).transpose(1, 2)

    return tok(T), tok(N * T), tok(N * T), tok(T)


def _ring_step(q, k, v, do, N, out, m, l, dq, dk, dv):
    """Forward, delta and backward through the operators, into given tensors."""
    ops = torch.ops.ring_attention_ops
    scale = 1.0 / math.sqrt(q.size(-1))
    m.fill_(float("-inf"))
    ops.ring_attention_forward(q, k, v, out, m, l, N, scale)
    D = ops.ring_attention_delta(do, out)
    ops.ring_attention_backward(q, dq, k, dk, v, dv, do, m, l, D, N, scale)


def _one_call_step(q, k, v, do, N):
    """The one-call operators, which allocate outputs and workspace themselves."""
    ops = torch.ops.ring_attention_ops
    scale = 1.0 / math.sqrt(q.size(-1))
    o, out, m, l = ops.ring_attention_attend(q, k, v, N, scale)
    return (o, out, m, l, *ops.ring_attention_grad(do, q, k, v, out, m, l, N, scale))


def _capture(step):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm-up outside capture, as torch requires
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static = step()
    return graph, static


# (H, T, chunks): whole grids; key pieces in forward and dQ and query splits in
# dK/dV, whose partials take the dQ partials' place in the workspace; the same
# of one chunk (the one-call operators' forward)
SHAPES = pytest.mark.parametrize("H,T,N,whole", [(2, 256, 2, True), (3, 1000, 2, False), (3, 1000, 1, False)])
HEAD_DIMS = pytest.mark.parametrize("D", [64, 128])  # compiled kernels; the hand-scheduled D = 128 loops


@SHAPES
@HEAD_DIMS
@pytest.mark.parametrize("one_call", [False, True])
def test_ring_attention_graph_replays_equal_eager(D, H, T, N, whole, one_call):
    harp_amd.load_ops()
    _lib.timing_enable(False)  # no per-launch timing events inside the capture
    plan = split_plan(1, H, T, D, N, T)
    assert plan == (1, 1, 1) if whole else min(plan[:2]) > N and plan[2] > 1
    q, k, v, do = _inputs(0, H=H, T=T, D=D, N=N)
    if one_call:
        names = ("o", "out", "m", "l", "dq", "dk", "dv")

        def step(q, k, v, do, outs):
            return _one_call_step(q, k, v, do, N)

        outs = None
    else:
        names = ("out", "m", "l", "dq", "dk", "dv")
        out = torch.empty(q.shape, dtype=torch.float32, device=DEV)
        m = torch.empty((1, H, T, 1), dtype=torch.bfloat16, device=DEV)
        l = torch.empty((1, H, T, 1), dtype=torch.float32, device=DEV)
        outs = (out, m, l, torch.empty_like(q), torch.empty_like(k), torch.empty_like(v))

        def step(q, k, v, do, outs):
            _ring_step(q, k, v, do, N, *outs)
            return outs

    graph, static = _capture(lambda: step(q, k, v, do, outs))
    for seed in (1, 2, 3):
        nq, nk, nv, ndo = _inputs(seed, H=H, T=T, D=D, N=N)
        for dst, src in ((q, nq), (k, nk), (v, nv), (do, ndo)):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in static]
        # eager on the same inputs, into fresh tensors
        ref = step(nq, nk, nv, ndo, outs and [torch.empty_like(t) for t in outs])
        torch.cuda.synchronize()
        for name, a, b in zip(names, got, ref):
            assert torch.equal(a, b), (seed, name)


def test_qk_norm_rope_graph_replays_equal_eager():
    harp_amd.load_async_ops()
    ops = torch.ops.async_op
    B, H, S, D = 1, 4, 128, 128
    g = torch.Generator().manual_seed(5)

    def tok():
        return torch.randn((B, S, H, D), generator=g).to(torch.bfloat16).to(DEV).transpose(1, 2)

    x, dy = tok(), tok()
    w = (1 + 0.1 * torch.randn(D, generator=g)).to(torch.bfloat16).to(DEV)
    ang = torch.arange(S, dtype=torch.float64)[:, None] * (10000.0 ** (-2.0 * torch.arange(D // 2) / D))[None, :]
    f = torch.polar(torch.ones_like(ang), ang).to(torch.complex64).to(DEV)
    y, dx = torch.empty_like(x), torch.empty_like(x)
    rms = torch.empty(B * H * S, dtype=torch.float32, device=DEV)
    gw = torch.empty(D, dtype=torch.bfloat16, device=DEV)

    def step(x_, dy_, y_, rms_, dx_, gw_):
        ops.qk_norm_rope_forward(x_, w, f, y_, rms_, 1e-6)
        ops.qk_norm_rope_backward(x_, dy_, w, rms_, f, dx_, gw_)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(x, dy, y, rms, dx, gw)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(x, dy, y, rms, dx, gw)

    for _ in range(3):
        nx, ndy = tok(), tok()
        x.copy_(nx)
        dy.copy_(ndy)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in (y, rms, dx, gw)]
        ref = [torch.empty_like(t) for t in (y, rms, dx, gw)]
        step(nx, ndy, *ref)
        torch.cuda.synchronize()
        for name, a, b in zip(("y", "rms", "dx", "grad_weight"), got, ref):
            assert torch.equal(a, b), name


def test_fused_producer_graph_replays_equal_eager():
    """The fused q/k/v projection kernel (harp_amd.qkv.qkv_project, with the
    pre-norm products and rms kept) at a shape whose half-empty last round
    goes to the tail launch: two launches in the graph."""
    from harp_amd import qkv

    B, S, dim, H = 1, 90 * 256, 128, 2
    g = torch.Generator().manual_seed(11)
    x = torch.randn((B, S, dim), generator=g).to(torch.bfloat16).to(DEV)
    ws = [(torch.randn((H * 128, dim), generator=g) / dim ** 0.5).to(torch.bfloat16).to(DEV) for _ in range(3)]
    w = (1 + 0.1 * torch.randn(128, generator=g)).to(torch.bfloat16).to(DEV)
    ang = torch.arange(S, dtype=torch.float64)[:, None] * (10000.0 ** (-2.0 * torch.arange(64) / 128))[None, :]
    f = torch.polar(torch.ones_like(ang), ang).to(torch.complex64).to(DEV)
    norms = [(w, 1e-6), (w, 1e-6), (None, 0.0)]

    def step(x_):
        outs, lins, rmss = qkv.qkv_project(x_, ws, norms, f, keep_for_backward=True)
        return list(outs) + [lins[0], lins[1], rmss[0], rmss[1]]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static = step(x)

    for _ in range(3):
        nx = torch.randn((B, S, dim), generator=g).to(torch.bfloat16).to(DEV)
        x.copy_(nx)
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in static]
        ref = step(nx)
        torch.cuda.synchronize()
        for name, a, b in zip(("q", "k", "v", "q_lin", "k_lin", "rms_q", "rms_k"), got, ref):
            assert torch.equal(a, b), name
