"""Host checks, no GPU: the choices of grid, tile and split by size (transformer_amd/csrc/plans.h, and the split counts that
the workspace queries show), at sizes that were measured on both sides of each rule."""
import ctypes

import pytest

from tests import plans

BASE, DEFAULT = 16, 14  # heads of the two layouts: 128 + 64 with a shared k_rope, 64 + 64 with one per head

# causal attention of B sequences of T: us in mirrored pairs and in single tiles, of the forward, and of the whole
# backward with one of its kernels changed (None: not measured).  Differences under 5 % are left out.
FORWARD = [(18, 448, DEFAULT, 32.7, 38.7), (20, 683, BASE, 81.8, 92.8), (6, 1500, DEFAULT, 58.8, 64.4),
           (12, 2048, BASE, 265, 279), (4, 2644, BASE, 180.6, 148.6), (3, 1608, BASE, 63.1, 51.6),
           (3, 1732, DEFAULT, 58.5, 44.9), (4, 1077, BASE, 49.9, 36.5), (2, 4729, DEFAULT, 216.2, 156.0),
           (3, 3000, BASE, 180, 144), (2, 2600, DEFAULT, 76, 63)]
DQ = [(1, 2928, DEFAULT, 139.4, 149.1), (18, 448, DEFAULT, 107.5, 112.8), (4, 1133, DEFAULT, 124.2, 113.4),
      (10, 387, BASE, 110.3, 99.2), (3, 1552, DEFAULT, 175.5, 153.8), (3, 1732, DEFAULT, 202.5, 176.7)]
DKDV = [(20, 709, BASE, 319.1, 337.7), (18, 448, DEFAULT, 107.5, 113.7), (20, 683, BASE, 302.5, 318.3),
        (1, 698, BASE, 67.8, 57.8), (3, 1452, BASE, 196.1, 162.4), (1, 486, BASE, 60.6, 49.2),
        (3, 1552, DEFAULT, 175.5, 138.7)]


@pytest.mark.parametrize("kernel,measured", [(0, FORWARD), (0, DQ), (1, DKDV)])
def test_attention_grids_take_the_faster_form_where_it_was_measured(kernel, measured):
    for B, T, H, pairs, single in measured:
        assert plans.single_tiles(B * H, T)[kernel] == (single < pairs), (B, T, H)


def test_one_tile_is_never_split_into_single_tiles():
    for n_bh in (1, 100, 257, 600, 5000):
        assert plans.single_tiles(n_bh, 128) == (False, False) and plans.single_tiles(n_bh, 1, False) == (False, False)


def test_norm_linear_tiles_at_measured_sizes():
    # us, wide / half / small tiles: 12288 x 2560 x 1792 129.0 / 146.0 / 168.8, 8192 x 2624 x 2048 132.8 / 127.7 / 140.7,
    # 2735 x 2000 x 1632 57.1 / 36.6 / 40.2, 1000 x 2624 x 2048 61.7 / 42.6 / 39.3
    for (M, N, K), kind in (((12288, 2560, 1792), plans.NL_WIDE), ((8192, 2624, 2048), plans.NL_HALF),
                            ((2735, 2000, 1632), plans.NL_HALF), ((1000, 2624, 2048), plans.NL_SMALL)):
        assert plans.norm_linear(M, N, K).kind == kind, (M, N, K)
    assert plans.norm_linear(24576, 2624, 2048) == (plans.NL_WIDE, 10, 960, 96)  # the last 64 columns apart


def test_norm_linear_tiles_cover_the_product_once():
    # n_wide tiles of n_nt columns, and a remainder's tiles only beside wide ones and for columns they do not cover
    tile = {plans.NL_WIDE: (256, 256), plans.NL_HALF: (256, 128), plans.NL_SMALL: (128, 128)}
    for M in (1, 127, 128, 129, 255, 257, 700, 6391, 14308, 24576):
        for N in (4, 96, 128, 132, 256, 260, 384, 388, 808, 868, 2500, 2624):
            for K in (32, 160, 2048):
                p = plans.norm_linear(M, N, K)
                bn, bm = tile[p.kind]
                mt = -(-M // bm)
                assert p.n_wide == mt * p.n_nt and p.n_rest in (0, mt)
                covered = p.n_nt * bn + (128 if p.n_rest else 0)
                assert N <= covered < N + bn and (not p.n_rest or (p.kind == plans.NL_WIDE and p.n_nt * bn < N))


def test_weight_grad_plans_cover_the_tokens_and_bound_the_workspace():
    for M in (1, 32, 33, 1000, 3001, 12288, 100000):
        for N, K in ((8, 8), (896, 384), (1792, 1792), (2560, 1792), (2056, 1800), (2624, 2048), (32768, 2048)):
            p = plans.weight_grad(M, N, K)
            tk = 128 if p.narrow else 256
            assert (p.nt, p.kt) == (-(-N // 256), -(-K // tk)) and p.seg % 32 == 0
            assert (p.S - 1) * p.seg < M <= p.S * p.seg
            assert p.part_bytes == (p.nt * p.kt * p.S * 256 * tk * 4 if p.S > 1 else 0) and p.part_bytes <= 256 << 20


def test_weight_grad_tiles_of_the_training_shapes():
    # the down-projections' gradients of one block's pass: wide tiles; weights with few tiles: narrow ones in segments
    assert not plans.weight_grad(12288, 2560, 1792).narrow and not plans.weight_grad(6150, 2624, 2048).narrow
    assert plans.weight_grad(12288, 896, 384) == (1, 21, 608, 4, 3, 33030144)
    assert plans.weight_grad(4100, 384, 1792).narrow


def _decode_workspace(B, L, H, d_latent, splits):
    from transformer_amd import _lib
    a = _lib.DecodeArgs()
    a.B, a.H, a.L, a.d_latent, a.d_rope, a.n_k_rope_heads, a.num_splits = B, H, L, d_latent, 64, 1, splits
    return int(_lib.entry("mla_decode_workspace_bytes")(ctypes.byref(a)))


def test_decode_splits_stay_within_one_round_of_the_cus():
    # us, rounded up -> down: B = 24 over 4000 45.7 -> 35.9, B = 40 over 3000 53.4 -> 40.4, B = 48 over 4000 77.6 -> 55.6,
    # B = 150 over 1000 71.5 -> 54.0.  The workspace holds the partials of every split, so it tells the counts apart
    for B, L in ((24, 4000), (40, 3000), (48, 4000), (32, 4096), (100, 2000)):
        assert _decode_workspace(B, L, 16, 512, 0) == _decode_workspace(B, L, 16, 512, 256 // B)
        assert _decode_workspace(B, L, 16, 512, 0) < _decode_workspace(B, L, 16, 512, 2 * (256 // B))
    assert _decode_workspace(150, 1000, 16, 512, 0) == _decode_workspace(150, 1000, 16, 512, 1)
    for B in (1, 3, 17, 24, 60, 129, 200, 256, 300):
        for H in (1, 16, 20):
            units = B * -(-H // 16)
            for d_latent in (128, 256, 384, 512):
                want = -(-256 // units) if d_latent == 128 else max(1, 256 // units)
                assert _decode_workspace(B, 20000, H, d_latent, 0) == \
                    _decode_workspace(B, 20000, H, d_latent, min(want, 20000 // 128)), (B, H, d_latent)


def _cached_plans(B, T, L0, H=16, d_latent=512):
    """The (waves a workgroup, key ranges) that the workspace fits: one record of 16 heads per query, padded to whole
    workgroups; empty for one range."""
    from transformer_amd import _lib
    a = _lib.PrefillCachedArgs()
    a.B, a.T, a.H, a.L0, a.L, a.d_latent, a.d_rope, a.num_splits = B, T, H, L0, L0 + T, d_latent, 64, 0
    total = int(_lib.entry("mla_prefill_cached_workspace_bytes")(ctypes.byref(a)))
    return [(nw, s) for nw in (4, 8) for s in range(2, 257)
            for recs in [B * -(-H // 16) * -(-T // nw) * nw * 16 * s]
            if -(-recs * d_latent * 4 // 256) * 256 + recs * 8 == total]


def test_cached_prefill_workgroups_and_ranges_at_measured_sizes():
    # us, before -> with these (16 heads, d_latent 512): B = 3, T = 100 over 2000 77.0 -> 54.7; B = 16, T = 100 over 1000
    # 117.7 -> 90.5 (one range); and T one past B = 1, T = 64 over 4000, where four waves took 34.4 and eight 40.2, and
    # B = 8, where they took 125.0 and 101.3 (T such that the two pad differently)
    assert _cached_plans(3, 100, 2000) == [(8, 6)]
    assert _cached_plans(16, 100, 1000) == []
    assert _cached_plans(1, 65, 4000) == [(4, 15)]
    assert _cached_plans(8, 65, 4000) == [(8, 3)]
