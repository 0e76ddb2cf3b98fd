"""How the attention kernels' keys are split between waves and blocks: the rules are plain functions of a step's sizes,
so what every kernel launch assumes of them is checked here for many sizes (the kernels refuse what breaks these,
`csrc/attention_mfma.hip` attention_launch: blocks of equally many shares for the decode kernel, a share that is a multiple of
32 keys, of 64 for the tiled kernel, and splits x share covering the longest context)."""
import itertools

import pytest

from inferrs_amd import ops


@pytest.mark.parametrize("g", [1, 2, 4, 5, 8, 16, 20])
def test_decode_split_covers_the_context_within_one_round_of_the_chip(g):
    for n_seqs, nkv, kv in itertools.product((1, 2, 3, 8, 16, 33, 64, 200), (1, 2, 8), (1, 31, 64, 500, 512, 513, 1024,
                                                                                     2048, 4096, 8192, 40960, 131072)):
        splits, chunk = ops.decode_split(n_seqs, nkv, g, kv)
        assert splits >= 1 and splits & (splits - 1) == 0 and splits <= 128
        assert chunk % 32 == 0 and splits * chunk >= kv
        if splits > 1:
            assert (splits - 1) * 32 < kv, "no more splits than steps of 32 keys (a split may be empty: shorter requests of a batch have such)"
            assert chunk >= 64, "a wave's share is worth two steps of 32 keys"
            items = n_seqs * nkv * -(-g // 16)
            assert items * splits <= ops.DECODE_WAVES, "one round of the chip"
        if kv <= 512:
            assert splits == 1 or chunk >= 128
        if splits > ops.DECODE_MANY_SPLITS:
            assert chunk > 64, "many blocks to merge only for long shares"


def test_decode_split_at_the_measured_points():
    # (32 query and 8 key/value heads; the choices that the measurements in the rule's description name)
    assert ops.decode_split(1, 8, 4, 8192)[0] == 64
    assert ops.decode_split(8, 8, 4, 8192)[0] == 16
    assert ops.decode_split(64, 8, 4, 8192)[0] == 2
    assert ops.decode_split(1, 8, 4, 2048)[0] == 32
    assert ops.decode_split(1, 8, 4, 1024)[0] == 16
    assert ops.decode_split(1, 8, 4, 512)[0] == 4
    assert ops.decode_split(2, 8, 4, 4096)[0] == 32


@pytest.mark.parametrize("d", [64, 128])
def test_prompt_split_covers_the_context(d):
    for n_seqs, nkv, g, q, kv in itertools.product((1, 3, 16), (1, 8), (1, 4, 5), (1, 2, 17, 128, 512, 2048),
                                                   (17, 512, 2048, 8192, 40000)):
        if q > kv:
            continue
        splits, chunk = ops.attention_split(n_seqs, nkv, g, q, kv, d)
        assert 1 <= splits <= 128 and splits * chunk >= kv and chunk % 32 == 0
        tiled = d == 128 and q * g >= ops.ATTN_TILE_COLS
        if tiled:
            assert chunk % 64 == 0, "the tiled kernel walks stages of 64 keys"
            if 2 * q > kv:
                assert splits == 1, "portions that span most of their context keep their keys together"


# Output features and k of the products of dense layers: width, feed-forward and query heads (of 128, beside 8 key heads).
DENSE = {"0.6B": (1024, 3072, 16), "1.7B": (2048, 6144, 16), "4B": (2560, 9728, 32), "8B": (4096, 12288, 32), "14B": (5120, 17408, 40),
         "32B": (5120, 25600, 64)}


@pytest.mark.parametrize("shape,product,rows,own", [
    # where whole steps were timed with the product on either kernel, on either side of the rule; narrow steps, which the host bounds
    # wherever they are met eagerly, stay with the kernel whose call costs less
    ("0.6B", "o", 512, True), ("0.6B", "down", 1000, True), ("0.6B", "o", 1024, False), ("0.6B", "down", 1024, False),
    ("1.7B", "o", 384, True), ("1.7B", "down", 900, True), ("1.7B", "o", 1024, False), ("1.7B", "down", 1024, True),
    ("4B", "o", 144, True), ("4B", "o", 420, True), ("8B", "down", 2048, True), ("8B", "o", 521, True), ("8B", "down", 200, True),
    ("14B", "down", 129, True), ("14B", "down", 1536, True), ("32B", "o", 1024, True)])
def test_products_behind_which_the_stream_is_normed_go_where_they_are_faster(shape, product, rows, own):
    width, ff, heads = DENSE[shape]
    assert bool(ops.library().ia_gemm_wide_norm_fits(rows, width, heads * 128 if product == "o" else ff)) == own


@pytest.mark.parametrize("shape,rows,own", [("0.6B", 512, True), ("0.6B", 1024, False), ("1.7B", 900, True), ("1.7B", 1024, False), ("4B", 409, True),
                                            ("4B", 410, False), ("4B", 640, False), ("8B", 160, True), ("8B", 456, True), ("8B", 1024, True),
                                            ("8B", 1025, False), ("14B", 521, True), ("14B", 900, True), ("32B", 456, True)])
def test_products_of_queries_and_keys_go_where_they_are_faster(shape, rows, own):
    width, _, heads = DENSE[shape]
    assert bool(ops.library().ia_gemm_wide_rope_fits(rows, (heads + 16) * 128, width)) == own


@pytest.mark.parametrize("shape,rows,own", [("0.6B", 512, True), ("0.6B", 700, True), ("1.7B", 456, True), ("4B", 160, True), ("4B", 580, True),
                                            ("4B", 768, False), ("4B", 900, True), ("8B", 200, True), ("8B", 320, True), ("8B", 456, False),
                                            ("8B", 512, False), ("8B", 700, True), ("14B", 130, False), ("14B", 200, False), ("14B", 521, False),
                                            ("14B", 832, True), ("14B", 1024, True), ("14B", 1025, False), ("32B", 1024, True)])
def test_gate_and_up_go_where_they_are_faster(shape, rows, own):
    width, ff, _ = DENSE[shape]
    assert bool(ops.library().ia_gemm_wide_dual_fits(rows, ff, width)) == own


def test_the_wide_kernels_rules_refuse_what_the_kernel_does_not_take():
    lib = ops.library()
    for fits in (lib.ia_gemm_wide_norm_fits, lib.ia_gemm_wide_rope_fits, lib.ia_gemm_wide_dual_fits):
        for m, n, k in ((0, 4096, 8192), (512, 0, 8192), (512, 4096, 0), (900, 8192, 8200), (900, 8194, 8192), (-5, -4, -64)):
            assert fits(m, n, k) == 0


def test_32_bit_products_of_up_to_8_rows_stay_on_the_vector_units():
    fits = ops.library().ia_gemm_f32_fits
    for n, k in ((6144, 4096), (24576, 4096), (65536, 2048), (128256, 4096), (151936, 1024), (151936, 4096), (262144, 2560)):
        assert not any(fits(m, n, k) for m in range(0, 9))
        assert all(fits(m, n, k) == (n >= 16384) for m in range(9, 17)) and fits(17, n, k) and not fits(17, n, k + 2)


@pytest.mark.parametrize("n,k,eight", [(131072, 2560, True), (151936, 4096, True), (151936, 1024, True), (131056, 1024, False), (128256, 4096, False)])
def test_a_logits_head_has_blocks_of_eight_waves_from_four_rounds_of_them_on(n, k, eight):
    """(`fills`: whether the plan's blocks are three stages deep, as those of eight waves are and the general ones are not)"""
    lib = ops.library()
    assert bool(lib.ia_gemm_mid_fills(n, k, 0)) == eight and lib.ia_gemm_mid_splits(n, k) == 1


def test_a_chunks_columns_are_shared_out_within_one_round_of_the_chip():
    """A chunk's block brings keys and queries of 64 tokens into shared memory: a compute unit holds two such blocks at 128 entries a
    key, three at 64, four (by their registers) at 32."""
    columns = ops.library().ia_linear_scan_columns
    for dim, at_once in ((128, 512), (96, 512), (64, 768), (32, 1024), (16, 1024)):
        for units, vt in itertools.product((1, 5, 100, 192, 255, 256, 257, 288, 320, 352, 384, 512, 513, 4000), (1, 32, 33, 64, 128, 161, 257)):
            cols = columns(units, vt, dim)
            shares = -(-vt // cols)
            assert cols >= 32 and cols % 32 == 0 and (shares == 1 or shares * units <= at_once), (dim, units, vt, cols)
    # (64 heads x 5 chunks, 32 x 11: two shares each would be a second round; 8 heads x 24 chunks: two shares, not three)
    assert columns(320, 64, 128) == 64 and columns(352, 64, 128) == 64 and columns(192, 257, 128) == 160 and columns(384, 128, 64) == 64


def test_bounds_of_mixed_steps_are_few_and_close():
    """A step of portions beside single tokens is captured once a pair of bounds: what bounds a run covers it, exceeds its bucket by a
    quarter at most (from eight buckets on), never exceeds the longer run's, and takes few values over a long prompt."""
    from inferrs_amd.engine import Engine
    bucket, widest = Engine.GRAPH_BUCKET_TOKENS, 40 * Engine.GRAPH_BUCKET_TOKENS
    for least, most in ((1, 17), (2, 16)):
        bounds = [Engine._run_bound(n, bucket, widest, least) for n in range(1, widest + 1)]
        for n, b in enumerate(bounds, 1):
            buckets = max(least, -(-n // bucket))
            assert n <= b <= widest and b % bucket == 0 and b // bucket <= buckets * 1.25
            assert buckets > 8 or b == buckets * bucket
        assert bounds == sorted(bounds) and len(set(bounds)) <= most
    assert Engine._run_bound(100, 1024, 1024, 2) == 1024 and Engine._run_bound(9000, 1024, 9 * 1024) == 9 * 1024
    # a portion of up to 2,048 tokens of context beside anything: one graph
    assert len({Engine._run_bound(n, bucket, widest, 2) for n in range(1, 2049)}) == 1


@pytest.mark.parametrize("heads,q_lens,kv_starts,span,plain,portions", [
    ((32, 8, 128), [555], [0], None, 309, 104), ((8, 8, 64), [144], [0], None, 26.3, 24.6), ((16, 2, 64), [17], [0], None, 16.8, 14.7),
    ((32, 8, 128), [16] * 16, [484] * 16, None, 339, 82), ((8, 8, 64), [64] * 16, [7936] * 16, None, 5956, 839),
    ((32, 4, 128), [2] * 64 + [500], [498] * 64 + [0], None, 405, 297), ((64, 8, 128), [5] * 73, [4700] * 73, None, 1859, 1079),
    ((8, 8, 64), [9] * 30, [4200] * 30, 19, 20.9, 66.6), ((16, 8, 128), [2] * 64 + [500], [3998] * 64 + [0], None, 1513, 9095),
    ((8, 8, 64), [3] * 32 + [512], [1997] * 32 + [2000], None, 886, 4331), ((16, 8, 128), [8] * 16, [492] * 16, None, 156, 281),
    ((8, 8, 64), [8] * 64, [7992] * 64, None, 2992, 6235), ((32, 8, 128), [2] * 16 + [200], [498] * 16 + [0], None, 170, 564),
    ((8, 8, 64), [16] * 16, [1984] * 16, None, 318, 757)])
def test_portions_in_32_bits_take_the_faster_kernel_at_the_measured_points(heads, q_lens, kv_starts, span, plain, portions):
    """The choice between the two 32-bit kernels as a layer makes it, against both measured times (us)."""
    from types import SimpleNamespace

    import torch
    from inferrs_amd.engine.batch import StepContext
    from inferrs_amd.parts.attention import Attention
    nq, nkv, d = heads
    spec = SimpleNamespace(n_heads=nq, n_kv_heads=nkv, head_dim=d, window=span, mask_chunk=None)
    ctx = SimpleNamespace(n_single=0, n_seqs=len(q_lens), n_tokens=sum(q_lens), q_lens=q_lens, kv_starts=kv_starts, _tables={},
                          max_kv_len=max(a + b for a, b in zip(q_lens, kv_starts)))
    ctx.once = lambda key, make: StepContext.once(ctx, key, make)
    q = torch.empty(0)
    assert Attention.portions_pay(spec, ctx, q) == (portions < plain)
    assert Attention.portions_pay(spec, ctx, q) == (portions < plain) and len(ctx._tables) == (len(q_lens) > 1)
    ctx.n_single = 1
    assert not Attention.portions_pay(spec, ctx, q) and not Attention.portions_pay(spec, SimpleNamespace(n_single=0), q.bfloat16())


@pytest.mark.parametrize("rows,n,k,dual,splits,tiles", [
    (24, 3072, 1024, 1, 1, 1), (117, 3072, 1024, 1, 1, 2), (64, 1024, 2048, 0, 4, 1), (117, 4096, 1024, 0, 2, 4),    # groups: two blocks a unit
    (103, 5120, 1024, 0, 2, 7), (107, 5120, 1536, 0, 2, 7), (84, 6144, 640, 1, 1, 6), (89, 8192, 512, 1, 1, 6),      # which these have no room for
    (64, 2560, 4096, 0, 8, 4), (117, 6144, 2048, 1, 1, 8), (16, 1024, 1024, 0, 2, 1),
    (73, 5120, 9728, 0, 1, 5), (75, 4096, 8192, 0, 1, 5), (86, 8192, 8192, 0, 1, 6),             # stored products, two stages: whole,
    (66, 1024, 4096, 0, 1, 1), (97, 4096, 8192, 0, 1, 2), (64, 4096, 8192, 0, 1, 1)])             # but for small weights and other rows
def test_rows_of_the_mid_products_are_grouped_within_one_round_of_the_chip(rows, n, k, dual, splits, tiles):
    """Tiles of 16 rows a block at measured points (256 compute units, which is what the rule takes without a GPU too)."""
    lib = ops.library()
    assert dual or splits == 1 or lib.ia_gemm_mid_splits(n, k) == splits
    assert lib.ia_gemm_mid_row_tiles(rows, n, k, dual, splits) == tiles


@pytest.mark.parametrize("n,k,splits", [(3200, 2048, 4), (3200, 3072, 4), (9728, 512, 1), (10240, 1152, 1),      # two stages are faster
                                        (3072, 1024, 2), (2560, 9728, 4), (1024, 3072, 4), (5120, 1536, 2), (3200, 3328, 2)])
def test_plans_of_small_weights_split_k_as_often_as_two_stages_would(n, k, splits):
    assert ops.library().ia_gemm_mid_splits(n, k) == splits


@pytest.mark.parametrize("g", [1, 2, 5, 8, 16, 20])
def test_decode_shares_are_whole_blocks_that_cover_the_context(g):
    """What a decode step takes in place of `decode_split`'s counts: as many waves as one round of the chip holds, blocks of equally
    many waves (up to four, so that more than four shares come in fours), shares of two steps of 32 keys or more."""
    others = set()
    for n_seqs, nkv, kv in itertools.product(range(1, 65), (1, 2, 4, 8), (31, 512, 513, 1024, 2048, 3072, 4095, 4096, 8192, 40960)):
        base = ops.decode_split(n_seqs, nkv, g, kv)
        for d, dv in ((64, 64), (128, 64), (128, 128), (192, 192), (256, 256)):
            splits, chunk = ops.decode_shares(n_seqs, nkv, g, kv, d, dv)
            assert chunk % 32 == 0 and splits * chunk >= kv and 1 <= splits <= 128
            assert splits <= 4 or splits % 4 == 0
            if (splits, chunk) != base:
                others.add((splits, max(d, dv)))
                assert chunk >= 64 and n_seqs * nkv * -(-g // 16) * splits <= ops.DECODE_WAVES
    widths = (64, 128, 192, 256)
    assert {w for s, w in others if s == 12} == {w for s, w in others if s == 28} == set(widths)
    assert {w for s, w in others if s == 4} == {64, 128}
    assert {w for s, w in others if s == 48} == (set(widths[:3]) if g <= 8 else set())
    assert {w for s, w in others if s == 64} == (set(widths[:3]) if g <= 4 else set())
    assert {s for s, _ in others} <= {4, 12, 28, 48, 64}


@pytest.mark.parametrize("n,nkv,g,d,dv,bound,span,kind,apart,fused", [
    (8, 4, 4, 128, 64, 2048, 1024, "gated", 15.5, 9.5), (8, 4, 4, 128, 64, 2048, 0, "gated", 16.2, 10.1), (1, 8, 2, 256, 256, 2048, 0, "gated", 17.8, 21.9),
    (16, 1, 16, 192, 192, 4096, 0, "plain", 22.0, 33.4), (1, 1, 16, 128, 128, 16384, 0, "gated", 16.2, 28.3), (24, 8, 2, 256, 256, 1024, 0, "plain", 43.5, 39.0),
    (64, 4, 4, 256, 256, 8192, 1024, "plain", 107.4, 69.2), (12, 8, 2, 64, 64, 8192, 1024, "plain", 19.8, 24.9), (24, 8, 2, 128, 128, 8192, 1024, "plain", 38.6, 29.4),
    (1, 4, 4, 128, 64, 8192, 0, "formed", 8.5, 11.1), (4, 4, 4, 128, 64, 4096, 1024, "formed", 8.8, 10.3), (9, 8, 5, 128, 128, 4096, 0, "formed", 27.4, 22.8),
    (64, 4, 4, 128, 64, 4096, 1024, "formed", 49.5, 25.1), (12, 8, 5, 128, 128, 8192, 1024, "formed", 22.5, 28.9), (1, 1, 16, 256, 256, 16384, 0, "formed", 15.4, 123.9),
    (2, 8, 2, 64, 64, 512, 0, "formed", 7.1, 5.5), (16, 2, 8, 128, 128, 1024, 0, "formed", 9.4, 9.7), (32, 2, 8, 128, 128, 1024, 0, "formed", 11.8, 10.5)])
def test_decode_attention_takes_the_faster_kernels_at_the_measured_points(n, nkv, g, d, dv, bound, span, kind, apart, fused):
    """The choice between one kernel and several as a layer makes it, against both measured times (us)."""
    assert ops.decode_fused_pays(n, nkv, g, d, dv, bound, span, formed=kind == "formed", gated=kind == "gated") == (fused < apart)


@pytest.mark.parametrize("m,n,k,own", [(800, 6144, 2560, 0), (900, 6144, 2560, 0), (800, 10240, 2560, 1), (1400, 6144, 2560, 1), (1300, 4096, 4096, 1),
                                       (2048, 4096, 4096, 0), (2048, 2560, 4096, 0), (2048, 4096, 1024, 0), (2047, 4096, 4096, 1), (1024, 8512, 2048, 1),
                                       (2048, 8512, 2048, 1), (511, 8512, 2048, 0)])
def test_whole_products_stay_with_the_vendor_where_nothing_is_gained(m, n, k, own):
    """Features in whole blocks of 256: up to 1,024 rows only where the plan is ahead clearly, and no multiples of 1,024 rows; odd ones as before."""
    assert ops.library().ia_gemm_wide_rows_fits(m, n, k) == own
