"""The fused q/k/v producer's smaller blocks (launch_proj in
harp_amd/csrc/proj_kernels.hip): 128 tokens x 1 head with four tiles in
flight, 128 x 2 heads with three, and both as parts of the large grid's last
units.  All sum in the same order as the large blocks, so every output is
compared bit for bit with a call that runs those (the same tokens repeated
until the grid fills the CUs), and the products with the fp64 product of the
same inputs (the bound of tests/test_gpu_qkv.py)."""

import math

import pytest
import torch

from harp_amd import qkv
from tests.test_gpu_qkv import _check_product, _inputs

pytestmark = pytest.mark.gpu

CUS = 256


def _route(S, heads, n_outs):
    tiles = n_outs * math.ceil(S / 128)
    if tiles * heads <= CUS:
        return "128x1"
    if tiles * ((heads + 1) // 2) <= CUS:
        return "128x2"
    per_out = math.ceil(S / 256) * ((heads + 1) // 2)
    units = n_outs * per_out
    r = units % CUS
    if not (0 < 2 * r <= CUS < units and r <= per_out):
        return "256x2"
    return "256x2+1" if 4 * r <= CUS else "256x2+2"


@pytest.mark.parametrize("S,dim,heads,n_outs,route", [
    (1, 64, 1, 1, "128x1"),        # one k-tile: three of the four stages stay empty
    (127, 128, 3, 3, "128x1"),     # two k-tiles, an odd head count, a partial tile
    (129, 320, 42, 3, "128x1"),    # five k-tiles (past the four stages), 252 blocks
    (257, 192, 29, 3, "128x2"),    # three k-tiles, one token in the last tile, half a last pair
    (640, 256, 34, 3, "128x2"),    # 255 blocks
    (641, 64, 34, 3, "256x2"),
    (140 * 256 - 130, 128, 3, 1, "256x2+1"),  # an odd last head and an empty second half in the tail
    (2048, 448, 30, 3, "256x2+2"),
])
def test_small_blocks_equal_large_blocks(S, dim, heads, n_outs, route):
    assert torch.cuda.get_device_properties(0).multi_processor_count == CUS
    assert _route(S, heads, n_outs) == route
    print(f"[S={S} dim={dim} heads={heads} outs={n_outs}: {route}]", flush=True)
    x, ws, norms, fc, _ = _inputs(1, S, dim, heads, "bf16", True, False, seed=S + dim)
    norms = (norms + [(None, 0.0)])[:n_outs]
    got = qkv.qkv_project(x, ws[:n_outs], norms, fc, keep_for_backward=True)
    # whole batches more, as rows of the same table, until no unit is left over for smaller blocks
    B = next(b for b in range(1, 1 << 16) if _route(b * S, heads, n_outs) == "256x2")
    want = qkv.qkv_project(x.expand(B, S, dim).contiguous(), ws[:n_outs], norms, fc, keep_for_backward=True)
    torch.cuda.synchronize()
    for i in range(n_outs):
        for b in (0, B - 1):
            assert torch.equal(got[0][i][0], want[0][i][b])
            if norms[i][0] is not None:
                assert torch.equal(got[1][i][0], want[1][i][b])
                assert torch.equal(got[2][i].view(heads, S), want[2][i].view(B, heads, S)[b])
        _check_product(x, ws[i], got[0][i] if norms[i][0] is None else got[1][i], f"out {i}")
