"""The attention kernels' grids: one tile per workgroup or mirrored pairs (TileGrid in mla_common.h), forward and backward
at sizes on both sides of each rule, against fp64 on the GPU, and bit for bit the same rows in either grid."""
import math

import pytest
import torch

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


@pytest.mark.parametrize("B,T,H,dn,hr", [
    (20, 300, 10, 64, 10),   # single tiles everywhere (400 pairs), three tiles, the last ragged
    (16, 257, 21, 128, 1),   # the same past a multiple of 8 (b, h), shared k_rope
    (8, 512, 16, 128, 1),    # dK/dV in pairs: one whole round of 256
    (1, 640, 3, 64, 3),      # few (b, h): dK/dV single, the forward's key split, dQ in pairs
])
def test_attention_grids_match_fp64(B, T, H, dn, hr):
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


def test_single_tiles_equal_pairs_bit_for_bit():
    # a batch whose grid runs single tiles against its sequences two at a time, whose grids run pairs or the key split
    # off (the forward's split merge rounds once more, so the forward is compared where neither splits)
    ops = torch.ops.mla_mi355x
    B, T, H = 20, 300, 10
    t, do = _inputs(B, T, H, 64, H, seed=1)
    scale = 0.1
    o, lse = ops.prefill_fwd(*t, scale, True, 0)
    grads = ops.prefill_bwd(do, *t, o, lse, scale, True, 0)
    for lo, hi in ((0, 13), (13, 20)):  # 260 and 140 pairs of q-tiles: more than 128, so no key split
        part = [v[lo:hi] for v in t]
        o2, lse2 = ops.prefill_fwd(*part, scale, True, 0)
        assert torch.equal(o2, o[lo:hi]) and torch.equal(lse2, lse[lo:hi])
        g2 = ops.prefill_bwd(do[lo:hi], *part, o2, lse2, scale, True, 0)
        assert all(torch.equal(a, b[lo:hi]) for a, b in zip(g2, grads))
