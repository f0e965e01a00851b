"""GPU: the RMSNorm / RoPE kernels on calls large enough for the walk (several
steps per block, two heads per unit with an odd H) against the same rows in
small calls (one step per block, one head per unit): each row's arithmetic is
the same, so the results are equal to the bit.  grad_weight against fp64."""

import pytest
import torch

import harp_amd

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
S, H, CUT = 7001, 9, 37  # 9 heads pair up as 5 + 4; 7001 tokens leave every grid a short last step


def _tensor(g, layout, B, D):
    if layout == "token":
        return torch.randn(B, S, H, D, device=DEV, generator=g).to(torch.bfloat16).transpose(1, 2)
    return torch.randn(B, H, S, D, device=DEV, generator=g).to(torch.bfloat16)


@pytest.mark.parametrize("layout", ["token", "head"])
@pytest.mark.parametrize("D", [40, 64, 72, 128, 200])
@pytest.mark.parametrize("op", ["norm_rope", "norm", "rope"])
def test_large_call_equals_small_calls(op, D, layout):
    harp_amd.load_async_ops()
    ops = torch.ops.async_op
    g = torch.Generator(device=DEV).manual_seed(D)
    B = 2 if D == 64 else 1
    x, dy = _tensor(g, layout, B, D), _tensor(g, layout, B, D)
    w = (1 + 0.1 * torch.randn(D, device=DEV, generator=g)).to(torch.bfloat16)
    ang = torch.rand(S, D // 2, device=DEV, generator=g) * 6.28
    f = torch.polar(torch.ones_like(ang), ang)

    def call(x, dy, f):
        y, dx = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
        rms = torch.full((x.numel() // D,), float("nan"), device=DEV)
        gw = torch.empty(D, device=DEV)
        if op == "rope":
            ops.rope_forward_impl(x, f, y)
            ops.rope_backward_impl(dy, f, dx)
        elif op == "norm":
            ops.rmsnorm_forward_out(x, w, y, rms, 1e-5)
            ops.rmsnorm_backward_out(x, dy, w, rms, dx, gw)
        else:
            ops.qk_norm_rope_forward(x, w, f, y, rms, 1e-5)
            ops.qk_norm_rope_backward(x, dy, w, rms, f, dx, gw)
        return y, dx, rms.view(x.shape[:3]), gw

    y, dx, rms, gw = call(x, dy, f)
    for a in (0, S // 2, S - CUT):
        part = call(x[:, :, a:a + CUT], dy[:, :, a:a + CUT], f[a:a + CUT])
        assert torch.equal(y[:, :, a:a + CUT], part[0]) and torch.equal(dx[:, :, a:a + CUT], part[1]), a
        assert op == "rope" or torch.equal(rms[:, :, a:a + CUT], part[2]), a
    assert not y.isnan().any() and not dx.isnan().any()
    if op == "rope":
        return
    g64 = dy.double()
    if op == "norm_rope":  # the RoPE backward, truncated to bf16 as the kernel's intermediate is
        c = torch.view_as_complex(g64.reshape(*dy.shape[:-1], -1, 2).contiguous()) * f.conj().to(torch.complex128)
        g32 = torch.view_as_real(c).flatten(-2).float()
        g64 = (g32.view(torch.int32) & -65536).view(torch.float32).double()
    ref = (g64 * x.double() / rms.double()[..., None]).sum((0, 1, 2))
    # fp32 sums of B*H*S terms, plus (norm_rope) single bf16 units of 2^-8
    # where fp64 and fp32 truncate apart: a few in 1e5 elements
    assert float((gw.double() - ref).norm() / ref.norm()) <= 1e-4


@pytest.mark.parametrize("D", [8, 24, 32, 40, 56, 64])
def test_row_sums_do_not_depend_on_the_lanes_per_row(D):
    """Rows of up to 64 elements (8 lanes each) against the same rows padded
    with zeros to four (D = 8: sixteen) times the length (16 lanes): the sum of
    squares is one fp32 tree, its mean differs by a power of four, so rms and y
    agree to the bit after scaling by that power's root."""
    harp_amd.load_async_ops()
    g = torch.Generator(device=DEV).manual_seed(D)
    x = torch.randn(1, 3, 2000, D, device=DEV, generator=g).to(torch.bfloat16)
    r = 4 if D == 8 else 2

    def norm(x, eps):
        y, rms = torch.empty_like(x), torch.empty(3 * 2000, device=DEV)
        w = torch.ones(x.size(-1), dtype=torch.bfloat16, device=DEV)
        torch.ops.async_op.rmsnorm_forward_out(x, w, y, rms, eps)
        return y, rms

    y, rms = norm(x, 2.0 ** -16)
    ypad, rpad = norm(torch.nn.functional.pad(x, (0, D * (r * r - 1))), 2.0 ** -16 / r ** 2)
    assert torch.equal(rms, rpad * r)
    assert torch.equal(y * r, ypad[..., :D])
