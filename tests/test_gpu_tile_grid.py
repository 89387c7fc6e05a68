"""The attention kernels' grids: one tile per workgroup or mirrored pairs (TileGrid in plans.h), forward and backward
at sizes on both sides of each rule, against fp64 on the GPU, and bit for bit the same rows in either grid."""
import math

import pytest
import torch

from tests import plans
from tests.gpu_util import check_close

pytestmark = pytest.mark.gpu


def _inputs(B, T, H, dn, hr, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    return [r(B, T, H, dn), r(B, T, H, 64), r(B, T, H, dn), r(B, T, hr, 64), r(B, T, H, 128)], r(B, T, H, 128)


def _fp64(t, do, scale, b, h):
    one = [v[b, :, min(h, v.size(2) - 1)].double().requires_grad_(True) for v in t]
    q, k = torch.cat(one[:2], -1), torch.cat(one[2:4], -1)
    s = (q @ k.t().contiguous()) * scale
    s = s.masked_fill(torch.ones_like(s).triu(1) > 0, float("-inf"))
    o = torch.softmax(s, -1) @ one[4]
    return o.detach(), torch.logsumexp(s, -1).detach(), torch.autograd.grad(o, one, do[b, :, h].double())


@pytest.mark.parametrize("B,T,H,dn,hr,single", [  # single: whether the forward and dQ, and dK/dV, run a tile a workgroup
    (20, 300, 10, 64, 10, (True, True)),   # three tiles, the last ragged
    (16, 257, 21, 128, 1, (True, True)),   # past a multiple of 8 (b, h), shared k_rope
    (8, 512, 16, 128, 1, (False, False)),  # dK/dV in pairs: one whole round of 256
    (1, 640, 3, 64, 3, (False, True)),     # few (b, h): the forward's key split, dQ in pairs
])
def test_attention_grids_match_fp64(B, T, H, dn, hr, single):
    assert plans.single_tiles(B * H, T) == single
    print(f"case B={B} T={T} H={H} dn={dn} hr={hr}", flush=True)
    ops = torch.ops.mla_mi355x
    t, do = _inputs(B, T, H, dn, hr)
    scale = 1 / math.sqrt(dn + 64)
    o, lse = ops.prefill_fwd(*t, scale, True, 0)
    grads = ops.prefill_bwd(do, *t, o, lse, scale, True, 0)
    for b, h in {(0, 0), (B - 1, H - 1), (B // 2, H // 2)}:
        ro, rl, rg = _fp64(t, do, scale, b, h)
        check_close(o[b, :, h].double().cpu(), ro.cpu(), f"o {b},{h}")
        torch.testing.assert_close(lse[b, h].double(), rl, rtol=0, atol=1e-3)
        for i, name in ((0, "dq_nope"), (1, "dq_rope"), (2, "dk_nope"), (4, "dv")):
            err = (grads[i][b, :, h].double() - rg[i]).norm() / rg[i].norm()
            assert err <= 1e-2, (name, b, h, float(err))


@pytest.mark.parametrize("B,part,T,H,dn,hr", [
    (13, 12, 400, 10, 64, 10),  # four tiles, the last ragged: 130 (b, h) run single tiles, 120 pairs
    (6, 5, 600, 17, 128, 1),    # five: 102 single, 85 pairs and a middle tile alone; shared k_rope
])
def test_single_tiles_equal_pairs_bit_for_bit(B, part, T, H, dn, hr):
    # a batch whose three kernels run single tiles against its first and last sequences, whose three kernels run pairs (more
    # than 128 of them, so the forward does not split its keys: its merge rounds once more)
    assert plans.single_tiles(B * H, T) == (True, True) and plans.single_tiles(part * H, T) == (False, False)
    assert part * H * ((T + 255) // 256) > 128
    ops = torch.ops.mla_mi355x
    t, do = _inputs(B, T, H, dn, hr, seed=1)
    scale = 0.1
    o, lse = ops.prefill_fwd(*t, scale, True, 0)
    grads = ops.prefill_bwd(do, *t, o, lse, scale, True, 0)
    for lo, hi in ((0, part), (B - part, B)):
        sub = [v[lo:hi] for v in t]
        o2, lse2 = ops.prefill_fwd(*sub, scale, True, 0)
        assert torch.equal(o2, o[lo:hi]) and torch.equal(lse2, lse[lo:hi])
        g2 = ops.prefill_bwd(do[lo:hi], *sub, o2, lse2, scale, True, 0)
        assert all(torch.equal(a, b[lo:hi]) for a, b in zip(g2, grads))
