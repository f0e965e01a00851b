"""GPU: calls whose grids leave most CUs idle, where the forward and dQ split
the keys of a chunk (not only the ring steps; harp_ra_forward of a single chunk
stays whole) and dK/dV splits the queries, against fp64 attention: piece edges, pad keys that leave pieces empty, several
chunks in rotated ring order, bf16 and fp32 gradients, unaligned bf16 views."""

import math

import pytest
import torch

import harp_amd
from harp_amd import ops as H_ops
from tests.gpu_harness import split_plan

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# (B, H, T, D, sp, chunk, valid per chunk, ring_rank)
SHAPES = [
    (1, 3, 1000, 128, 1, 1000, [1000], 0), (1, 2, 511, 128, 1, 4096, [4000], 0), (1, 2, 513, 128, 3, 700, [700, 129, 0], 1),
    (2, 1, 2049, 128, 2, 513, [513, 257], 1), (1, 3, 1000, 64, 1, 1000, [999], 0), (1, 2, 576, 64, 3, 600, [600, 1, 300], 2),
    (1, 2, 700, 72, 2, 1030, [1030, 512], 0), (1, 2, 640, 96, 1, 900, [900], 0), (1, 1, 2000, 40, 2, 520, [520, 520], 1),
]


def _ref(q, k, v, dout, keep):
    q, k, v, dout = (t.double() for t in (q, k[:, :, keep], v[:, :, keep], dout))
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    p = torch.softmax(s, -1)
    o = torch.matmul(p, v)
    ds = p * (torch.matmul(dout, v.transpose(-1, -2).contiguous()) - (dout * o).sum(-1, keepdim=True)) * scale
    return (o, torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2).contiguous(), q),
            torch.matmul(p.transpose(-1, -2).contiguous(), dout), torch.logsumexp(s, -1))


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("B,H,T,D,sp,chunk,lens,rank", SHAPES)
@pytest.mark.parametrize("grads", ["bf16", "fp32", "bf16 unaligned"])
def test_split_calls_against_fp64(B, H, T, D, sp, chunk, lens, rank, grads):
    _, dq_splits, dkdv_splits = split_plan(B, H, T, D, sp, chunk, lens)
    assert dq_splits > sp and (dkdv_splits > 1) == (T >= 576)  # 513 queries: two splits don't pay
    if grads == "bf16 unaligned" and D == 128:
        pytest.skip("head dim 128 stores bf16 gradients 8 bytes at a time: the C ABI refuses such views")
    g = torch.Generator(device=DEV).manual_seed(T + D)
    q, dout = (torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    k, v = (torch.randn(B, sp * chunk, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    pos = torch.arange(sp * chunk, device=DEV)
    keep = (pos % chunk) < torch.tensor(lens, device=DEV)[pos // chunk]
    o64, dq64, dk64, dv64, lse64 = _ref(q, k, v, dout, keep)
    scale = 1.0 / math.sqrt(D)
    kc = [k[:, :, c * chunk:(c + 1) * chunk] for c in range(sp)]
    vc = [v[:, :, c * chunk:(c + 1) * chunk] for c in range(sp)]
    out, m, l = torch.empty_like(q, dtype=torch.float32), torch.empty(B, H, T, device=DEV), torch.empty(B, H, T, device=DEV)
    H_ops.abi_forward(q, kc, vc, out, m, l, scale, rank, lens)
    delta = torch.empty(B, H, T, device=DEV)
    H_ops.abi_delta(dout, out, delta)
    dt = torch.float32 if grads == "fp32" else torch.bfloat16
    pad = 1 if "unaligned" in grads else 0  # rows start on odd elements
    mk = lambda n: torch.full((B, n, H, D + pad), float("nan"), device=DEV, dtype=dt)[..., pad:].transpose(1, 2)  # noqa: E731
    dq, dk, dv = mk(T), mk(sp * chunk), mk(sp * chunk)
    ch = lambda t: [t[:, :, c * chunk:(c + 1) * chunk] for c in range(sp)]  # noqa: E731
    H_ops.abi_backward(q, dq, kc, vc, ch(dk), ch(dv), dout, m, l, delta, scale, rank, lens)
    assert float((m.double() + l.double().log() - lse64).abs().max()) <= 1e-4
    # P, dS and (bf16 outputs) the results are rounded to bf16, 2^-9 rms each:
    # at most three such roundings reach a result
    for name, a, b in (("o", out, o64), ("dq", dq, dq64), ("dk", dk[:, :, keep], dk64), ("dv", dv[:, :, keep], dv64)):
        assert _rel(a, b) <= 3 * 2.0 ** -9, (name, _rel(a, b))
    assert not dk[:, :, ~keep].any() and not dv[:, :, ~keep].any()


def test_a_smaller_workspace_keeps_whole_grids():
    """A workspace for the statistics alone (all that whole grids need) is
    taken; a smaller one is refused."""
    lib = harp_amd.load_abi()
    B, H, T, D = 1, 2, 1024, 128
    need, stats = H_ops.backward_workspace_bytes(B, H, T, D, 1, T), 2 * 4 * H * T
    assert need > stats  # split partials
    assert H_ops.forward_workspace_bytes(B, H, T, D, 1, T) > 0
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v, dout = (torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(4))
    o64, dq64, dk64, dv64, _ = _ref(q, k, v, dout, torch.ones(T, dtype=torch.bool, device=DEV))
    out, delta = torch.empty_like(q, dtype=torch.float32), torch.empty(B, H, T, device=DEV)
    m, l = torch.empty_like(delta), torch.empty_like(delta)
    scale = 1.0 / math.sqrt(D)
    none = torch.empty(0, dtype=torch.uint8, device=DEV)  # a NULL workspace
    H_ops.abi_forward(q, [k], [v], out, m, l, scale, workspace=none)
    H_ops.abi_delta(dout, out, delta)
    grads = [torch.empty_like(q) for _ in range(3)]

    def backward(nbytes):
        ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        H_ops.abi_backward(q, grads[0], [k], [v], [grads[1]], [grads[2]], dout, m, l, delta, scale, workspace=ws)

    for nbytes in (stats, need - 256, need):
        for t in grads:
            t.fill_(float("nan"))
        backward(nbytes)
        for name, a, b in (("o", out, o64), ("dq", grads[0], dq64), ("dk", grads[1], dk64), ("dv", grads[2], dv64)):
            assert _rel(a, b) <= 3 * 2.0 ** -9, (name, nbytes, _rel(a, b))
    with pytest.raises(RuntimeError, match="workspace"):
        backward(stats - 256)
    assert "smaller" in lib.harp_ra_last_error().decode()


def test_a_plan_below_the_ring_steps_runs_without_a_workspace():
    """Two short chunks and many queries: dK/dV splits the queries in less
    memory than two dQ splits by ring steps would take.  That plan runs with a
    workspace of exactly its size and, from the library's buffer, with none."""
    B, H, T, D, chunk = 1, 8, 2048, 128, 64
    need = H_ops.backward_workspace_bytes(B, H, T, D, 2, chunk)
    stats, ring = 2 * 4 * B * H * T, 2 * 4 * B * H * T + 2 * 4 * B * H * T * D
    assert stats < need < ring and (need - stats) % (B * H * 2 * chunk * 8 * D) == 0
    g = torch.Generator(device=DEV).manual_seed(3)
    q, dout = (torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    k, v = (torch.randn(B, 2 * chunk, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    o64, dq64, dk64, dv64, _ = _ref(q, k, v, dout, torch.ones(2 * chunk, dtype=torch.bool, device=DEV))
    ch = lambda t: [t[:, :, c * chunk:(c + 1) * chunk] for c in range(2)]  # noqa: E731
    out, delta = torch.empty_like(q, dtype=torch.float32), torch.empty(B, H, T, device=DEV)
    m, l = torch.empty_like(delta), torch.empty_like(delta)
    scale = 1.0 / math.sqrt(D)
    H_ops.abi_forward(q, ch(k), ch(v), out, m, l, scale)
    H_ops.abi_delta(dout, out, delta)

    def backward(nbytes):
        grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        H_ops.abi_backward(q, grads[0], ch(k), ch(v), ch(grads[1]), ch(grads[2]), dout, m, l, delta, scale, workspace=ws)
        return grads

    for nbytes in (need, 0):  # 0: a NULL workspace
        for name, a, b in zip(("dq", "dk", "dv"), backward(nbytes), (dq64, dk64, dv64)):
            assert _rel(a, b) <= 3 * 2.0 ** -9, (name, nbytes, _rel(a, b))
    assert all(torch.equal(a, b) for a, b in zip(backward(need), backward(0)))
    with pytest.raises(RuntimeError, match="workspace"):
        backward(need - 256)


@pytest.mark.parametrize("D", [64, 128])
def test_forward_of_one_chunk_leaves_its_workspace_alone(D):
    """harp_ra_forward of one chunk needs no workspace: a buffer that is passed
    all the same is neither written nor refused for its alignment, so calls on
    several streams may be handed the same one."""
    B, H, T = 1, 2, 1024
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(3))
    nbytes = H_ops.forward_workspace_bytes(B, H, T, D, 1, T)
    assert nbytes > 0  # the size at which harp_ra_forward_rounded splits the keys
    buf = torch.full((nbytes + 512,), 0x5a, dtype=torch.uint8, device=DEV)
    res = []
    for ws in (torch.empty(0, dtype=torch.uint8, device=DEV), buf, buf[8:]):
        out, m, l = torch.empty_like(q, dtype=torch.float32), torch.empty(B, H, T, device=DEV), torch.empty(B, H, T, device=DEV)
        H_ops.abi_forward(q, [k], [v], out, m, l, 1.0 / math.sqrt(D), workspace=ws)
        res.append((out, m, l))
    assert bool((buf == 0x5a).all())
    for r in res[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, res[0]))


@pytest.mark.parametrize("B,H,T,D,sp,chunk,lens,rank", SHAPES)
def test_one_call_operators_on_small_grids(B, H, T, D, sp, chunk, lens, rank):
    """The same shapes through ring_attention_attend / ring_attention_grad,
    which split the keys of a single chunk too: the rounded output stored by
    the merge, D formed by each key piece's dQ block."""
    harp_amd.load_ops()
    ops = torch.ops.ring_attention_ops
    assert (split_plan(B, H, T, D, sp, chunk, lens)[0] > sp) == (T != 2049)  # 2049: 770 keys a tile don't pay
    g = torch.Generator(device=DEV).manual_seed(T + D)
    q, dout = (torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    k, v = (torch.randn(B, sp * chunk, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2) for _ in range(2))
    pos = torch.arange(sp * chunk, device=DEV)
    keep = (pos % chunk) < torch.tensor(lens, device=DEV)[pos // chunk]
    o64, dq64, dk64, dv64, lse64 = _ref(q, k, v, dout, keep)
    scale = 1.0 / math.sqrt(D)
    o, out, m, l = ops.ring_attention_attend(q, k, v, sp, scale, rank, lens, chunk)
    assert torch.equal(o, out.to(torch.bfloat16))
    only, none, m1, l1 = ops.ring_attention_attend(q, k, v, sp, scale, rank, lens, chunk, False)
    assert torch.equal(only, o) and none.numel() == 0 and torch.equal(m1, m) and torch.equal(l1, l)
    dq, dk, dv = ops.ring_attention_grad(dout, q, k, v, out, m, l, sp, scale, rank, lens, chunk)
    assert float(((m.double() + l.double().log()).squeeze(-1) - lse64).abs().max()) <= 1e-4
    # as test_split_calls_against_fp64
    for name, a, b in (("o", out, o64), ("dq", dq, dq64), ("dk", dk[:, :, keep], dk64), ("dv", dv[:, :, keep], dv64)):
        assert _rel(a, b) <= 3 * 2.0 ** -9, (name, _rel(a, b))
    assert not dk[:, :, ~keep].any() and not dv[:, :, ~keep].any()
