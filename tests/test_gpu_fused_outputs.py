"""GPU: the one-call operators (ring_attention_attend / ring_attention_grad)
against the separate ones they replace: the rounded output is bf16(out) to the
bit, and so are the gradients: D formed in the dQ kernel is summed in
ring_attention_delta's order."""

import math

import pytest
import torch

import harp_amd
from tests.gpu_harness import split_plan

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# (D, B, H, T, sp, chunk, valid): staged and unstaged epilogues, one row, tile
# edges, a split over the chunks (3 heads, 8 chunks), pad keys; key pieces and
# query splits: tests/test_gpu_small_grids.py
SHAPES = [
    (64, 1, 2, 1, 1, 40, 40), (64, 2, 3, 257, 4, 130, 130), (72, 1, 2, 255, 2, 200, 190),
    (96, 1, 2, 256, 1, 128, 128), (96, 1, 2, 129, 3, 64, 50), (104, 1, 2, 33, 2, 70, 70),
    (128, 1, 2, 1, 1, 32, 32), (128, 1, 3, 255, 8, 96, 96), (128, 2, 2, 257, 1, 300, 300), (128, 1, 30, 256, 8, 64, 60),
]


def _view(g, B, H, T, D):
    return torch.randn(B, T, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2)


@pytest.mark.parametrize("D,B,H,T,sp,chunk,valid", SHAPES)
@pytest.mark.parametrize("keep", [True, False])
def test_one_call_operators_match_the_separate_ones(D, B, H, T, sp, chunk, valid, keep):
    harp_amd.load_ops()
    ops = torch.ops.ring_attention_ops
    g = torch.Generator(device=DEV).manual_seed(D * 1000 + T)
    q, dout = _view(g, B, H, T, D), _view(g, B, H, T, D)
    k, v = _view(g, B, H, sp * chunk, D), _view(g, B, H, sp * chunk, D)
    lens = None if valid == chunk else [valid] * sp
    assert (H, sp) != (3, 8) or split_plan(B, H, T, D, sp, chunk, lens) == (8, 8, 1)
    scale = 1.0 / math.sqrt(D)
    out = torch.empty_like(q, dtype=torch.float32)
    m = torch.empty(B, H, T, 1, device=DEV, dtype=torch.bfloat16)
    l = torch.empty(B, H, T, 1, device=DEV)
    ops.ring_attention_forward(q, k, v, out, m, l, sp, scale, 0, lens, chunk)
    o1, out1, m1, l1 = ops.ring_attention_attend(q, k, v, sp, scale, 0, lens, chunk, keep)
    assert o1.dtype == torch.bfloat16 and o1.stride() == q.stride()
    assert torch.equal(o1, out.to(torch.bfloat16))
    assert torch.equal(m1, m) and torch.equal(l1, l)
    if not keep:
        assert out1.numel() == 0
        return
    assert torch.equal(out1, out) and out1.stride() == out.stride()
    delta = ops.ring_attention_delta(dout, out)
    grads = [torch.empty_like(t) for t in (q, k, v)]
    ops.ring_attention_backward(q, grads[0], k, grads[1], v, grads[2], dout, m, l, delta, sp, scale, 0, lens, chunk)
    fused = ops.ring_attention_grad(dout, q, k, v, out1, m1, l1, sp, scale, 0, lens, chunk)
    for name, a, b in zip(("dq", "dk", "dv"), fused, grads):
        assert a.stride() == b.stride(), name
        # two orders of a D-term fp32 sum differ by < D * 2^-24 of its terms:
        # that moves single bf16 results (one unit, 2^-8 of the value) only
        err = float((a.double() - b.double()).norm() / b.double().norm())
        assert err <= 2.0 ** -10, (name, err)
    assert torch.equal(fused[2], grads[2])  # dV does not read D


# every head dim variant of the dQ kernels, D of up to 16 chunks of 8 elements
@pytest.mark.parametrize("D", [8, 16, 40, 64, 72, 80, 96, 104, 128])
def test_in_kernel_rowsum_is_bit_equal_to_the_delta_operator(D):
    """ring_attention_grad's gradients equal those of ring_attention_delta +
    ring_attention_backward bit for bit (fp32 sums of other orders moved 1 in
    10^4 to 10^5 of the bf16 results, so some of these would differ)."""
    harp_amd.load_ops()
    ops = torch.ops.ring_attention_ops
    g = torch.Generator(device=DEV).manual_seed(D)
    B, H, T, L = 1, 16, 513, 640
    q, dout, k, v = _view(g, B, H, T, D), _view(g, B, H, T, D), _view(g, B, H, L, D), _view(g, B, H, L, D)
    scale = 1.0 / math.sqrt(D)
    _, out, m, l = ops.ring_attention_attend(q, k, v, 1, scale)
    delta = ops.ring_attention_delta(dout, out)
    grads = [torch.empty_like(t) for t in (q, k, v)]
    ops.ring_attention_backward(q, grads[0], k, grads[1], v, grads[2], dout, m, l, delta, 1, scale)
    fused = ops.ring_attention_grad(dout, q, k, v, out, m, l, 1, scale)
    for name, a, b in zip(("dq", "dk", "dv"), fused, grads):
        assert torch.equal(a, b), (name, int((a != b).sum()))


def test_rows_of_an_unwritten_output_do_not_reach_others():
    """A NaN row of dO reaches only its own query's dQ through the in-kernel D."""
    ops = torch.ops.ring_attention_ops
    harp_amd.load_ops()
    g = torch.Generator(device=DEV).manual_seed(5)
    B, H, T, D = 1, 2, 70, 128
    q, k, v, dout = (_view(g, B, H, T, D) for _ in range(4))
    o, out, m, l = ops.ring_attention_attend(q, k, v, 1, 1.0 / math.sqrt(D))
    clean = ops.ring_attention_grad(dout, q, k, v, out, m, l, 1, 1.0 / math.sqrt(D))[0]
    bad = dout.clone()
    bad[0, 1, 69, 3] = float("nan")
    dq = ops.ring_attention_grad(bad, q, k, v, out, m, l, 1, 1.0 / math.sqrt(D))[0]
    assert bool(dq[0, 1, 69].isnan().all())
    keep = torch.ones(B, H, T, dtype=torch.bool, device=DEV)
    keep[0, 1, 69] = False
    assert torch.equal(dq[keep], clean[keep])
