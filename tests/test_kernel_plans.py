"""The host-side plans of the attention kernels stay inside what the kernels take (no GPU needed)."""

import pathlib
import re

import pytest

from conftest import ROOT


def test_key_shares_never_exceed_what_the_merge_takes():
    from tie_amd import kernels

    header = (pathlib.Path(ROOT) / "tiny-inference-engine_amd" / "csrc" / "attention_merge.h").read_text()
    assert int(re.search(r"#define\s+MERGE_MAX_SPLITS\s+(\d+)", header).group(1)) == kernels.MAX_KEY_SPLITS
    contexts = [1, 100, 1024, 4096, 32768, 40960, 65536, 131072, 1 << 20]
    for seqs in (1, 2, 3, 4, 7, 8, 64, 256):
        for kv_heads in (1, 2, 4, 8, 16):
            for context in contexts:
                for block_size in (4, 8, 16, 64):
                    n = kernels.decode_splits(seqs, kv_heads, context, block_size)
                    assert 1 <= n <= kernels.MAX_KEY_SPLITS, (seqs, kv_heads, context, block_size, n)
    # the cases that used to ask for more than the kernel takes
    assert kernels.decode_splits(1, 4, 65536, 8) == kernels.MAX_KEY_SPLITS
    assert kernels.decode_splits(1, 2, 81920, 8) == kernels.MAX_KEY_SPLITS
    assert kernels.decode_splits(1, 1, 65536, 16) == kernels.MAX_KEY_SPLITS
    # about 512 waves in shares of at least 128 keys where a wave keeps several tiles in flight
    assert kernels.decode_splits(8, 8, 4096) == 8 and kernels.decode_splits(64, 8, 4096) == 1
    assert kernels.decode_splits(31, 8, 4096) == 3 and kernels.decode_splits(32, 8, 4096) == 1 and kernels.decode_splits(48, 8, 4096) == 2
    assert kernels.decode_splits(1, 8, 4096) == 32 and kernels.decode_splits(1, 8, 200) == 1
    # where 512 waves would not spread evenly over 256 compute units, the count up to twice as large that does
    assert kernels.decode_splits(24, 8, 4096) == 4 and kernels.decode_splits(40, 8, 4096) == 3      # 768 and 960 waves
    assert kernels.decode_splits(12, 8, 4096) == 8 and kernels.decode_splits(20, 8, 4096) == 6      # 768 and 960
    assert kernels.decode_splits(24, 8, 300) == 2 and kernels.decode_splits(56, 8, 4096) == 2       # short shares; 1344 are too many
    # whatever the batch: between the count for 512 waves and twice that, more shares than that count only where
    # the GPU holds all their waves at once, and shares of at least 128 keys
    for seqs in range(1, 130):
        for kv_heads in (1, 2, 4, 8):
            for context in (200, 1024, 4096, 40000):
                n = kernels.decode_splits(seqs, kv_heads, context)
                pairs = seqs * kv_heads
                first = min(-(-512 // pairs), max(1, context // 128), kernels.MAX_KEY_SPLITS)
                assert (n == 1 and pairs == 256) or first <= n <= 2 * first, (seqs, kv_heads, context, n)
                assert n == 1 or context // n >= 64, (seqs, kv_heads, context, n)
                assert n <= first or pairs * n <= 1024, (seqs, kv_heads, context, n)
    for items in (1, 2, 5, 40, 300):
        for kv_heads in (1, 2, 8):
            for group in (1, 3, 4, 8, 16):
                for context in contexts:
                    n = kernels.prefill_splits(items, kv_heads, group, context, 64 * items)
                    assert 1 <= n <= kernels.MAX_KEY_SPLITS, (items, kv_heads, group, context, n)
    # one workgroup on each CU: a second beside it for long contexts that are read, and only for those
    assert [kernels.prefill_splits(32, 8, 2, context, 2048) for context in (1024, 2047, 2048, 16000)] == [1, 1, 2, 2]
    assert kernels.prefill_splits(32, 8, 2, 16000, 2048, 512) == 1 and kernels.prefill_splits(33, 8, 2, 16000, 2112) == 1
    # beside waves of single rows: never more shares than alone, few workgroups as alone, 64 and more cut for 256 places
    for items in (1, 4, 8, 16, 40):
        for context in (64, 500, 1181, 2000, 16000):
            alone = kernels.prefill_splits(items, 8, 2, context, 64 * items)
            beside = kernels.prefill_splits(items, 8, 2, context, 64 * items, beside_waves=True)
            assert 1 <= beside <= alone and (items >= 8 or beside == alone) and (beside == 1 or items * 8 * beside <= 256 or items < 8)
    assert [kernels.prefill_splits(n, 8, 2, c, 64 * n, beside_waves=True) for n, c in ((8, 1181), (8, 2000), (16, 1000), (8, 500))] \
        == [2, 4, 2, 2]


def test_float32_attention_cuts_keys_while_all_workgroups_run_at_once():
    """At most 256 workgroups where there is more than one share, no share empty, none of fewer than eight tiles of 16 keys
    but by what rounding leaves, at most 24 shares; the measured choices. The context is the end of a bucket that a recorded
    step serves: one sequence of 100 keys in sixteen shares of 1024 took a layer 1.0 us more than in four."""
    from tie_amd import kernels

    for tiles in (1, 2, 4, 5, 8, 16, 31, 32, 33, 301):
        for kv_heads, group in ((8, 2), (4, 8), (1, 40), (2, 16)):
            workgroups = tiles * kv_heads * -(-group // 16)
            for context in (1, 16, 17, 64, 65, 129, 300, 601, 1000, 4096, 33000):
                n, key_tiles = kernels.attention_f32_splits(tiles, kv_heads, group, context), -(-context // 16)
                share = -(-key_tiles // n)
                assert 1 <= n <= 24 and (n == 1 or workgroups * n <= 256), (tiles, kv_heads, group, context, n)
                assert share * (n - 1) < key_tiles and (n == 1 or share >= 5), (tiles, kv_heads, group, context, n)
    assert [kernels.attention_f32_splits(1, 8, 2, c) for c in (64, 128, 129, 300, 1024, 2048, 4096)] == [1, 1, 2, 3, 8, 16, 24]
    assert [kernels.attention_f32_splits(t, 8, 2, 1024) for t in (1, 2, 4, 8, 16, 32, 38)] == [8, 8, 8, 4, 2, 1, 1]


def test_sizes_no_kernel_takes_are_refused_when_the_model_is_built():
    from tie_amd.config.qwen3 import Qwen3Config
    from tie_amd.errors import InvalidArgument
    from tie_amd.models import Model
    from tie_amd.models.qwen3 import build_qwen3_spec
    from conftest import TINY_A

    with pytest.raises(InvalidArgument, match="head_dim 520"):
        Model(build_qwen3_spec(Qwen3Config.from_json(dict(TINY_A, head_dim=520))))
    Model(build_qwen3_spec(Qwen3Config.from_json(dict(TINY_A, head_dim=512))))


def test_the_cache_has_a_precision_of_its_own_where_a_kernel_takes_the_pair():
    """float32 arithmetic runs over float32, bfloat16 or float16 pages (the reference's KVCacheConfig.dtype,
    src/kv/paged_kv_cache.h:18-25); the matrix-core kernels read bfloat16 pages only. What no kernel takes is
    refused when the engine is made, by name, before any weight is read."""
    from tie_amd import kernels
    from tie_amd.api import create_engine
    from tie_amd.engine.replay import TraceReplayer
    from tie_amd.errors import InvalidArgument

    assert kernels.cache_dtype_for("float32") == "float32" and kernels.cache_dtype_for("bfloat16") == "bfloat16"
    assert kernels.cache_dtype_for("float32", "bf16") == "bfloat16"
    assert kernels.cache_dtype_for("float32", "float16") == "float16"
    assert kernels.cache_dtype_for("bfloat16", "bfloat16") == "bfloat16"
    for mode, asked, words in (("bfloat16", "float32", "bfloat16 arithmetic over a float32 cache"),
                               ("bfloat16", "float16", "bfloat16 arithmetic over a float16 cache"),
                               ("float32", "int8", "float32, bfloat16 or float16")):
        with pytest.raises(InvalidArgument, match=words):
            kernels.cache_dtype_for(mode, asked)
    # the folder does not exist: the refusal comes first
    with pytest.raises(InvalidArgument, match="over a float32 cache"):
        create_engine("/nonexistent/model", dtype="bfloat16", kv_dtype="float32")
    with pytest.raises(InvalidArgument, match="over a float16 cache"):
        TraceReplayer.from_folder("/nonexistent/model", "bfloat16", 64, kv_dtype="float16")


def test_cache_pages_are_sized_by_the_cache_dtype():
    from tie_amd.cache.manager import CacheManager
    from tie_amd.config.qwen3 import Qwen3Config
    from tie_amd.errors import InvalidArgument
    from tie_amd.models import Model
    from tie_amd.models.qwen3 import build_qwen3_spec
    from conftest import TINY_A

    plan = Model(build_qwen3_spec(Qwen3Config.from_json(TINY_A))).cache_plan
    sizes = {d: CacheManager(plan, block_size=4, num_blocks=8, dtype=d).bytes_per_block
             for d in ("float32", "bfloat16", "float16")}
    assert sizes["float32"] == 2 * sizes["bfloat16"] == 2 * sizes["float16"] == 2 * 2 * 2 * 4 * 16 * 4
    with pytest.raises(InvalidArgument, match="int8"):
        CacheManager(plan, block_size=4, num_blocks=8, dtype="int8")


TILE_ROWS_COLS = {4: (256, 256), 5: (256, 128), 6: (128, 256), 7: (128, 128), 10: (256, 192), 11: (128, 192)}


def test_the_tiled_product_plans_by_rounds_of_workgroups():
    """Above 128 rows the tile and the ranges of K come from an estimate of the time; these are the measured choices."""
    from tie_amd import kernels

    qkv, o, gate_up, down = (6144, 4096), (4096, 4096), (24576, 4096), (4096, 12288)    # [N, K] of an 8B layer
    # 2048 rows, the prefill step that is measured: 256 x 256 tiles; O alone is too narrow for them and stays whole;
    # QKV's 6144 columns in tiles of 192 make 256 workgroups where tiles of 256 leave a quarter of the compute
    # units idle (88 against 93 us)
    assert (kernels.gemm_tile(2048, *qkv, True), kernels.gemm_splits(2048, *qkv, True)) == (10, 1)
    assert (kernels.gemm_tile(2048, *o, True), kernels.gemm_splits(2048, *o, True)) == (6, 1)
    assert kernels.gemm_tile(2048, *gate_up, True, 1) == 4
    assert (kernels.gemm_tile(2048, *down, True), kernels.gemm_splits(2048, *down, True)) == (4, 2)
    assert kernels.gemm_splits(1024, *down, True) == 4
    # 768 rows: two ranges of 256 x 128 tiles would be 288 workgroups, a second round for 32 of them
    tile, ranges = kernels.gemm_tile(768, *qkv, True), kernels.gemm_splits(768, *qkv, True)
    rows, cols = TILE_ROWS_COLS[tile]
    assert -(-768 // rows) * -(-6144 // cols) * ranges <= 256
    # every plan: a tile that loads straight into LDS, 1 to 8 ranges, none shorter than 512 of K
    for N, K in (qkv, o, down, (2048, 2048), (10240, 5120), (5120, 25600)):
        for M in range(129, 2300, 61):
            ranges = kernels.gemm_splits(M, N, K, True)
            assert ranges in (1, 2, 4, 8) and (ranges == 1 or K // ranges >= 512), (M, N, K, ranges)
            assert kernels.gemm_tile(M, N, K, True) in TILE_ROWS_COLS
            assert kernels.gemm_tile(M, N, K, True, 1) in TILE_ROWS_COLS
    # 65 to 128 rows: the weights are read once, and one round of workgroups should fill the compute units.
    # 8B gate/up on 128 x 128 tiles (192 workgroups; 96 of 128 x 256 took 82 us against 61), the 1.7B's on
    # 64 x 128 (192), the 32B's on 128 x 256 (200); the 32B's QKV in 4 ranges (160 workgroups; 8 are two rounds)
    assert kernels.gemm_tile(128, *gate_up, True, 1) == 7 and kernels.gemm_tile(80, *gate_up, True, 1) == 7
    assert kernels.gemm_tile(96, 12288, 2048, True, 1) == 9 and kernels.gemm_tile(128, 51200, 5120, True, 1) == 6
    assert (kernels.gemm_tile(128, 10240, 5120, True), kernels.gemm_splits(128, 10240, 5120, True)) == (6, 4)
    assert (kernels.gemm_tile(128, 4096, 2048, True), kernels.gemm_splits(128, 4096, 2048, True)) == (9, 4)
    assert (kernels.gemm_tile(128, *down, True), kernels.gemm_splits(128, *down, True)) == (7, 8)
    for N, K in (qkv, o, down, (2048, 2048), (10240, 5120), (5120, 25600), (2048, 6144)):
        for M in range(65, 129, 9):
            ranges = kernels.gemm_splits(M, N, K, True)
            assert ranges in (1, 2, 4, 8) and (ranges == 1 or K // ranges >= 512), (M, N, K, ranges)
            assert kernels.gemm_tile(M, N, K, True) in (6, 7, 8, 9) and kernels.gemm_tile(M, N, K, True, 1) in (6, 7, 8, 9)
    # shapes the straight-to-LDS tiles do not take keep the older tiles and their rule
    assert kernels.gemm_splits(300, 200, 1000) == 2 and kernels.gemm_tile(300, 200, 1000) == 1
    assert kernels.gemm_splits(128, 4096, 4096) == 8 and kernels.gemm_splits(128, 4096, 256) == 1


@pytest.mark.parametrize("tile,splits,M,N,K,past", [
    (7, 4, 128, 4096, 4096, True), (7, 4, 128, 4080, 4096, False), (7, 4, 129, 4096, 4096, False), (9, 8, 64, 4096, 4096, True),
    (9, 8, 65, 4096, 4096, False), (6, 1, 100, 51200, 5120, True), (8, 1, 40, 65520, 3072, True), (10, 1, 256, 24576, 4096, False),
    (11, 2, 512, 6144, 4096, True), (11, 1, 256, 24576, 4096, True), (11, 1, 512, 12288, 2048, True), (11, 4, 256, 3072, 8192, True),
    (11, 1, 160, 24576, 4096, True), (11, 1, 450, 10240, 5120, False),
    (11, 1, 200, 19456, 2560, False), (11, 1, 200, 17920, 1536, False), (11, 1, 400, 10240, 5120, False),
    (11, 1, 900, 5120, 3072, False), (11, 1, 1107, 4096, 2048, False), (11, 1, 1200, 3584, 3584, False), (11, 1, 3000, 6144, 4096, False)])
def test_packed_weights_go_past_the_caches_where_they_are_read_once(tile, splits, M, N, K, past):
    """One row tile of 64 or 128 rows over 32 MB and more; on 128 x 192 row tiles that run beside each other on one die: tiles
    a multiple of eight, at most eight of them along M, the last one full enough for the length of a range. Those at the end
    took 3 to 10 us longer past the caches."""
    from tie_amd import kernels

    assert kernels.gemm_weights_past_caches(M, N, K, tile, splits) == past


@pytest.mark.parametrize("tile,splits,M,N,K,last", [
    (7, 1, 512, 2048, 2048, False), (7, 4, 128, 2048, 2048, False), (7, 4, 512, 2048, 2048, True), (7, 2, 400, 4096, 2048, True),
    (9, 4, 120, 2048, 2048, False), (9, 8, 120, 2048, 6144, False), (9, 4, 120, 2000, 2048, False), (9, 4, 120, 2064, 2048, True),
    (7, 4, 256, 1024, 3072, False), (7, 4, 200, 3584, 3584, False), (7, 4, 160, 4096, 4096, False), (7, 2, 300, 4096, 2048, False),
    (7, 8, 160, 2048, 6144, True), (4, 4, 600, 4096, 12288, True), (11, 2, 300, 2560, 4096, True), (10, 2, 700, 3584, 18944, True)])
def test_ranges_of_k_come_last_where_a_die_then_reads_less(tile, splits, M, N, K, last):
    """Tiles that are no multiple of eight, four row tiles and more, or ranges that spare a die 1.5 MB of x. Elsewhere the
    order by tiles is the faster one, by up to 1.6 us a product (256 rows over 1024 x 3072, 200 over 3584 x 3584)."""
    from tie_amd import kernels

    assert kernels.gemm_ranges_last(M, N, K, tile, splits) == last


@pytest.mark.parametrize("M,N,K,want", [(2048, 4096, 12288, (1, 5)), (2048, 4096, 4096, (1, 5)), (2048, 2048, 6144, (2, 5)),
                                        (512, 4096, 12288, (4, 5)), (512, 2048, 2048, (4, 7))])
def test_products_that_add_to_the_stream_have_a_plan_of_their_own(M, N, K, want):
    """The best of all forced (ranges, tile), each timed with the norm behind it, or within 2 % of it; every plan is one the
    kernel takes: no range shorter than 512 of K, and up to 128 rows the same as of products that store."""
    from tie_amd import kernels

    assert kernels.gemm_adding_plan(M, N, K) == want
    for rows in list(range(129, 2300, 61)) + [65, 100, 128, 48]:
        ranges, tile = kernels.gemm_adding_plan(rows, N, K)
        assert ranges in (1, 2, 4, 8) and (ranges == 1 or K // ranges >= 512), (rows, N, K, ranges)
        if rows > 128:
            assert tile in TILE_ROWS_COLS
        else:
            assert (ranges, tile) == (kernels.gemm_splits(rows, N, K, True), kernels.gemm_tile(rows, N, K, True))


def test_the_tiled_product_plans_for_a_last_row_tile_that_is_nearly_empty():
    """A nearly empty last row tile makes the others faster, tiles that are no multiple of eight slower: the best of all
    forced (tile, ranges) at 576, 320 and 144 rows, by 3 to 20 % (4096 x 12288 at 576 rows: 128 x 192 tiles in two
    ranges take 98 us with the kernel that adds the planes, 256 x 256 in four 81)."""
    from tie_amd import kernels

    for M, N, K, want in ((576, 4096, 12288, (4, 4)), (576, 8192, 8192, (4, 2)), (576, 8192, 28672, (4, 2)),
                          (320, 5120, 17408, (7, 2)), (144, 3072, 8192, (7, 4))):
        assert (kernels.gemm_tile(M, N, K, True), kernels.gemm_splits(M, N, K, True)) == want, (M, N, K)
    assert kernels.gemm_tile(576, 19456, 2560, True, 1) == 4


def test_the_common_launch_takes_what_its_library_says(monkeypatch):
    """Heads of 32, 64 and 128 over pages of 16, 32, ... positions; what the kernel's library answers is the rule."""
    from tie_amd import kernels

    for Dh in (16, 32, 48, 64, 96, 128, 256, 20):
        for bs in (4, 8, 12, 16, 32, 48, 64):
            assert kernels.attention_mixed_takes(Dh, bs) == (Dh in (32, 64, 128) and bs in (16, 32, 64)), (Dh, bs)
    asked = []
    monkeypatch.setattr(kernels, "_lib", lambda key, Dh=0: type("L", (), {"tie_attention_mixed_takes": staticmethod(lambda bs: asked.append((Dh, bs)) or 0)}))
    kernels.attention_mixed_takes.cache_clear()
    assert not kernels.attention_mixed_takes(128, 16) and asked == [(128, 16)]
    kernels.attention_mixed_takes.cache_clear()


def test_single_rows_beside_portions_share_their_keys_by_their_own_launch(monkeypatch):
    """32 sequences of 8 KV heads, a wave to a whole sequence where they run alone. In one launch with a portion (heads of 128)
    they are cut in two, unless a window leaves them less than two shares of 128 keys; heads of 256 have a launch of their own,
    and its plan, in the same step."""
    import torch

    from tie_amd import kernels

    shares = []
    monkeypatch.setattr(kernels, "attention_mixed_bf16", lambda *a, **k: shares.append(("mixed", k["single_nsplit"])))
    monkeypatch.setattr(kernels, "attention_decode_bf16", lambda *a, **k: shares.append(("decode", a[11])))
    monkeypatch.setattr(kernels, "attention_prefill_bf16", lambda *a, **k: None)
    S, KVH, bs = 32, 8, 16

    class Step:
        block_tables = torch.zeros(S + 1, 256, dtype=torch.int32)

    def scratch(name, shape, dtype):
        return torch.empty(0)

    for order in ((128, 256), (256, 128)):
        class Batch:
            all_decode, num_seqs, plan_context, memo = False, S + 1, 4096, {}
            host_new_tokens, host_context_lens = [64] + [1] * S, [64] + [4000] * S
            query_start = context_lens = seq_of_row = None

        shares.clear()
        for Dh in order:
            for window in (None, 128):
                H = KVH * 2
                q = torch.empty(S + 64, H * Dh, dtype=torch.bfloat16)
                cache = torch.empty(1, KVH, bs, Dh, dtype=torch.bfloat16)
                kernels.paged_attention(q, cache, cache.transpose(2, 3), torch.empty_like(q), Step, Batch, H, Dh ** -0.5, window, scratch)
        want = {128: [("mixed", 2), ("mixed", 1)], 256: [("decode", 1), ("decode", 1)]}
        assert shares == want[order[0]] + want[order[1]], (order, shares)


def test_float32_products_of_many_rows_take_pieces():
    """(rows, w): float32 instructions up to 32 rows over every w and to about 130 over 2048 x 2048, bfloat16 pieces above, from
    fewer rows the larger w is; K beyond a descriptor's reach stays on the former."""
    from tie_amd import kernels

    for M, N, K, pieces in ((4, 2048, 2048, False), (64, 4096, 2048, False), (48, 2048, 6144, False), (200, 4096, 2048, True),
                            (301, 2048, 6144, True), (301, 2048, 2048, True), (1000, 12288, 2048, True),
                            (1000, 64, (1 << 22) + 4, False)):
        splits = kernels.gemm_f32_splits(M, N, K)
        assert (kernels.gemm_f32_shape(M, N, K, splits) > 8) == pieces, (M, N, K)
        assert splits in (1, 2, 4, 8)
    assert kernels.gemm_f32_shape(301, 12288, 2048) == 10 and kernels.gemm_f32_shape(48, 12288, 2048) <= 8


@pytest.mark.parametrize("M,N,K,powers", [(301, 4096, 2048, (12, 10, 10)), (180, 6144, 4096, (5, 10, 10)), (350, 3072, 3072, (5, 10, 10)),
                                          (530, 4096, 2048, (10, 10, 10))])
def test_float32_products_in_three_ranges(M, N, K, powers):
    """Where three ranges of K fill a round of workgroups better than powers of two: tiles of 256 columns on pieces, ranges of
    at least 384 of K, all workgroups at once on the fullest die too, and a caller that fixes 1, 2 or 4 ranges gets that
    number's shape."""
    from tie_amd import kernels

    assert kernels.gemm_f32_splits(M, N, K) == 3 and K // 3 >= 384
    shape = kernels.gemm_f32_shape(M, N, K, 3)
    assert shape in (9, 10) and -(-M // 64) * -(-3 * N // (8 * 256)) <= 32 * (2, 1)[shape - 9]
    assert tuple(kernels.gemm_f32_shape(M, N, K, splits) for splits in (1, 2, 4)) == powers


@pytest.mark.parametrize("M,N,K", [(400, 3072, 2048), (440, 3072, 2048), (420, 3072, 3072), (380, 6144, 2560), (600, 4096, 2048),
                                   (350, 7168, 5120), (720, 7168, 5120), (850, 3072, 8192), (470, 5120, 3072)])
def test_float32_products_are_not_cut_in_three_for_a_second_round(M, N, K):
    """A die takes whole pieces of w: three ranges that leave one of them with more workgroups than run at once took up to
    1.4 times as long (400 rows over 3072 x 2048, 35 on a die of 32 compute units: 68.6 us, in two ranges 50.1)."""
    from tie_amd import kernels

    assert kernels.gemm_f32_splits(M, N, K) in (1, 2, 4, 8)


@pytest.mark.parametrize("N,K,rows", [(4096, 4096, {301: 8, 513: 8, 600: 8}), (6144, 4096, {140: 8, 321: 8, 384: 8, 400: 4, 700: 4}),
                                      (4096, 12288, {300: 8, 529: 8, 600: 8, 900: 8}), (4096, 2048, {301: 4, 513: 4, 587: 4, 640: 4}),
                                      (2048, 6144, {600: 8}), (5120, 5120, {220: 8, 400: 8, 500: 8, 800: 4}),
                                      (3072, 3072, {641: 8, 700: 4}), (7168, 5120, {160: 8, 270: 8, 350: 4, 600: 4})])
def test_float32_products_in_three_ranges_sum_in_no_fewer_chains(N, K, rows):
    """Beside the chains of sums (groups of waves along K, times ranges of K) of the best choice among powers of two: three
    ranges, where they are taken, have as many at least. The error of a sum grows with the length of its chains."""
    from tie_amd import kernels

    for M, chains in rows.items():
        splits = kernels.gemm_f32_splits(M, N, K)
        shape = kernels.gemm_f32_shape(M, N, K, splits)
        assert shape > 8 and (1, 2, 1, 2)[shape - 9] * splits >= chains, (M, N, K, splits, shape, chains)


def test_float32_products_run_on_what_was_fastest():
    """Up to 32 rows no weight takes pieces, in however many ranges of K. (rows, w): the choices within a tenth of the fastest
    one that was timed."""
    from tie_amd import kernels

    weights = ((512, 3072), (1024, 1024), (2048, 2048), (4096, 2048), (2048, 6144), (2560, 9728), (6144, 4096), (12288, 2048),
               (12288, 4096), (24576, 4096), (32000, 2048), (32000, 6144), (151936, 2048))
    for M in (1, 2, 3, 4, 5, 8, 16, 17, 24, 32):
        for N, K in weights:
            for splits in (kernels.gemm_f32_splits(M, N, K), 1, 2, 8):
                assert kernels.gemm_f32_shape(M, N, K, splits) <= 8, (M, N, K, splits)
    for M, N, K, good in ((5, 2048, 2048, {(2, 8), (1, 4), (1, 2)}), (16, 2048, 2048, {(2, 8), (1, 4), (1, 2), (2, 4)}),
                          (16, 151936, 2048, {(2, 1), (2, 2)}), (8, 151936, 2048, {(1, 1), (2, 2)}),
                          (5, 151936, 2048, {(1, 1), (2, 2)}), (5, 32000, 2048, {(1, 1), (2, 2)}),
                          (24, 12288, 4096, {(6, 4), (4, 2), (4, 4), (6, 8), (6, 1)}), (128, 4096, 2048, {(8, 2)}),
                          (64, 6144, 4096, {(12, 4), (9, 8), (10, 8)}), (200, 4096, 2048, {(9, 4), (10, 4), (12, 2)})):
        splits = kernels.gemm_f32_splits(M, N, K)
        assert (kernels.gemm_f32_shape(M, N, K, splits), splits) in good, (M, N, K, kernels.gemm_f32_shape(M, N, K, splits), splits)


def test_float32_products_of_one_to_four_rows_on_multiply_adds():
    """One and two rows over w of 1024 rows and more. Three and four over w of 64 MB whose rows are shorter than 16 KB: the
    kernel on multiply-adds is about as fast there and the more exact one. Rows of 16 KB took it up to a tenth longer."""
    from tie_amd import kernels

    for N, K, more in ((2048, 2048, False), (4096, 4096, False), (12288, 2048, True), (19456, 2560, True), (12288, 4096, False),
                       (24576, 4096, False), (151936, 2048, True), (5120, 640, False)):
        for M in (1, 2, 3, 4, 5):
            assert (kernels.gemm_f32_shape(M, N, K, 1) < 0) == (M <= 2 or more and M <= 4), (M, N, K)
    assert kernels.gemm_f32_shape(1, 512, 3072, 1) > 0


def test_float32_products_on_pieces_sum_in_enough_chains():
    """A product on pieces (shapes 9 to 12: one or two groups of waves along K, times the ranges of K) in fewer than two chains
    is further off than the float32 instructions', which have four at least (2.3e-7 and 1.7e-7 of a sum of 2048 numbers of
    one sign)."""
    from tie_amd import kernels

    seen = 0
    for N, K in ((512, 3072), (2048, 2048), (4096, 2048), (2048, 6144), (12288, 2048), (24576, 4096), (2560, 9728), (4096, 1000)):
        for M in (33, 64, 100, 128, 200, 256, 301, 512, 700, 1000, 2000):
            for splits in (kernels.gemm_f32_splits(M, N, K), 1, 2):
                shape = kernels.gemm_f32_shape(M, N, K, splits)
                seen += shape > 8
                assert shape <= 8 or (1, 2, 1, 2)[shape - 9] * splits >= 2, (M, N, K, splits, shape)
    assert seen > 100


def test_experts_take_wide_row_tiles_where_these_still_fill_the_gpu():
    """(experts, inner size): rows of a tile at 40, 100, 200, 400 and 600 rows an expert. Many or wide experts take 256
    from 192 on, smaller sets from 480 (16 experts of 512 at 384 rows: 41 us in tiles of 128, 56 in tiles of 256)."""
    import torch
    from tie_amd import kernels

    for real, inner, want in ((64, 1536, [64, 128, 256, 256, 256]),
                              (32, 768, [64, 128, 128, 128, 256]), (16, 512, [64, 128, 128, 128, 256]),
                              (64, 256, [64, 128, 128, 128, 128]), (192, 256, [64, 128, 256, 256, 256])):
        got = [kernels.moe_tile_rows(torch.bfloat16, torch.bfloat16, 1024, inner, n * real, real, packed=True)
               for n in (40, 100, 200, 400, 600)]
        assert got == want, (real, inner)


def test_the_prefill_attention_kernel_refuses_caches_it_cannot_address():
    """Its addresses are 32-bit counts of 8 bytes, a page's number times the page's size by a 24-bit multiply."""
    import torch
    from tie_amd import kernels

    def plane(pages, kv_heads, block, dim):
        return torch.empty((pages, kv_heads, block, dim), dtype=torch.bfloat16, device="meta")

    assert kernels.prefill_addressable(plane(300_000, 8, 16, 128))          # 9.8 GB: a long cache of an 8B model
    assert kernels.prefill_addressable(plane((1 << 20) - 1, 8, 16, 128))    # just under 32 GB
    assert not kernels.prefill_addressable(plane(1 << 20, 8, 16, 128))      # 32 GB
    assert not kernels.prefill_addressable(plane(4, 64, 4096, 256))         # a page of 128 MB
    assert not kernels.prefill_addressable(plane(1 << 24, 1, 4, 16))        # 2^24 pages


def test_the_decode_products_plan_for_17_to_64_rows():
    """Which kernel, how many tiles a workgroup and how many ranges of K come from one score (what x costs beside
    the weights, the planes, how full the compute units are), not from a table of shapes: its choices on the shapes
    it was measured on, and what must hold on any shape."""
    from tie_amd import kernels

    # 8B QKV at 24 rows: x through LDS, three tiles a workgroup, two ranges: 256 workgroups, one a compute unit
    # (15.1 us with the kernel that adds the planes; six tiles in four ranges, the same 256 workgroups: 17.1)
    assert kernels.few_rows_plan(24, 6144, 4096) == (True, 3, 2)
    # a gate/up of 16384 x 3072: 1024 tiles are 342 workgroups of three or 171 of six, a round and a third or two
    # thirds of one; x from memory in workgroups of four tiles fills one round exactly (20.6 against 22.4 and 24.7 us)
    assert kernels.few_rows_plan(24, 16384, 3072, True) == (False, 4, 1)
    # a gate/up of 34816 x 5120: eight tiles a workgroup would be 272 workgroups, a second round for 16 of them
    assert kernels.few_rows_plan(32, 34816, 5120, True) == (True, 3, 1)
    # up to 16 rows the shape alone decides
    assert kernels.few_rows_plan(16, 6144, 4096) == (False, 0, kernels.skinny_splits(6144, 4096))
    for N, K in ((6144, 4096), (4096, 12288), (5120, 3072), (2560, 9728), (1024, 2048), (8192, 28672), (10240, 5120)):
        for M in (17, 24, 32, 33, 48, 64):
            shares_x, tiles, splits = kernels.few_rows_plan(M, N, K)
            assert splits in (1, 2, 4, 8) and tiles in ((3, 6, 8) if shares_x else (1, 2, 3, 4)), (M, N, K)
            if shares_x:      # whole chunks of four k-blocks a wave, ranges of at least 1024 of K
                assert (K // 32) % (16 * splits) == 0 and (splits == 1 or K // splits >= 1024), (M, N, K, splits)
            assert kernels.few_rows_plan(M, N, K, True)[2] == 1                      # a gated product is never cut
    # the tiled product with 64-row tiles: the 32B shape's QKV in two ranges of 64 x 128 tiles (160 workgroups), not
    # eight of 64 x 256 (320: a second round for 64 of them, 1.7 times the time); a tile is the same whether the
    # plan is asked for the ranges too or handed them back
    assert (kernels.gemm_tile(64, 10240, 5120, True), kernels.gemm_splits(64, 10240, 5120, True)) == (9, 2)
    for N, K in ((6144, 4096), (4096, 12288), (10240, 5120), (8192, 8192), (1024, 2048), (5120, 25600)):
        for M in (40, 64):
            ranges = kernels.gemm_splits(M, N, K, True)
            assert ranges in (1, 2, 4, 8) and (ranges == 1 or K // ranges >= 512)
            assert kernels.gemm_tile(M, N, K, True) == kernels.gemm_tile(M, N, K, True, ranges) in (8, 9)
    assert kernels.gemm_tile(64, 51200, 5120, True, 1) == 8 and kernels.gemm_tile(64, 151936, 4096, True, 1) == 8


def test_portions_give_way_to_single_rows_that_bring_more():
    from tie_amd import kernels

    spread = [1900 // 16 + (1900 - 1900 // 16) * i // 30 for i in range(31)]
    assert kernels.portions_give_way(spread, 8, 1181)
    assert kernels.portions_give_way(spread, 8, 2048) and not kernels.portions_give_way(spread, 8, 2049)   # late portions
    assert not kernels.portions_give_way([350] * 28, 8, 1181)          # little to bring
    assert kernels.portions_give_way([32 * 16] * 32, 8, 700) and not kernels.portions_give_way([32 * 16] * 32, 4, 700)
    assert not kernels.portions_give_way([32 * 16] * 31 + [32 * 15], 8, 700)
    assert not kernels.portions_give_way([20000] * 32, 8, 700, reach=480)      # as much as the window shows


def test_sequences_of_different_lengths_stay_whole_where_no_compute_unit_waits_for_another():
    """Waves of whole sequences against shares of one length: by the tiles of the busiest compute unit, for head sizes that
    were measured, and only where every sequence is one wave's."""
    import random

    from tie_amd import kernels

    def spread(n, longest):
        return [max(1, longest // 16 + (longest - longest // 16) * i // (n - 1)) for i in range(n)]

    rng = random.Random(3)
    at_random = [max(1, int(2500 * rng.random() ** 2)) for _ in range(80)]
    assert kernels.decode_share_plan(spread(64, 1500), 8, 2048, head_dim=128) == (1, 0)
    assert kernels.decode_share_plan(spread(32, 500), 16, 1024, head_dim=64) == (1, 0)
    assert kernels.decode_share_plan([1500] * 20 + [500] * 44, 8, 2048, head_dim=128) == (1, 0)
    # long sequences that meet on one unit; heads that were not better or not searched; nothing known
    assert kernels.decode_share_plan(at_random, 8, 4096, head_dim=128)[1] > 0
    assert kernels.decode_share_plan([2000] * 8 + ([100] * 24 + [2000] * 8) + [100] * 24, 8, 2048, head_dim=128)[1] > 0
    for head_dim in (0, 16, 32, 256):
        assert kernels.decode_share_plan(spread(64, 1500), 8, 2048, head_dim=head_dim) == (8, 17)
    # one wave a unit (256 pairs), and sequences cut into shares of their own: the same plan for every head size
    for lens, heads in ((spread(32, 3000), 8), (at_random[:56], 8), ([4000] * 14 + [800] * 42, 8), (at_random, 4), (at_random + at_random[:20], 6)):
        plans = {kernels.decode_share_plan(lens, heads, 4096, head_dim=d) for d in (0, 64, 96, 128, 256)}
        assert len(plans) == 1 and plans.pop()[1] > 0, (len(lens), heads)
    # in a window a sequence has no more tiles than the window shows
    assert kernels.decode_share_plan([100] * 8 + [30000] * 56, 8, 32768, window=1024, head_dim=128) == (1, 0)


@pytest.mark.parametrize("S,heads", [(64, 8), (90, 8), (129, 4), (64, 16), (86, 6), (512, 1), (2, 300)])
def test_whole_sequences_are_launched_so_that_long_ones_meet_short_ones(S, heads):
    """A permutation; with sequences of lengths at random the busiest compute unit brings little more than the mean where
    every unit has the same number of waves. Without whole sequences, and below two waves a unit, there is no order; the plan
    for sequences of any length keeps the shares that the rule for them gives unless whole ones in order fill the units."""
    import random

    from tie_amd import kernels

    rng = random.Random(S)
    lens = [rng.randint(50, 2000) for _ in range(S)]
    tiles = kernels.key_tiles(lens)
    order = kernels.whole_sequences_order(tiles, heads)
    assert sorted(order.tolist()) == list(range(S)) and order.dtype.name == "int32"
    apart = max(1, 256 // heads)
    if S % apart == 0 and S > apart:
        assert kernels.whole_sequences_fill([tiles[i] for i in order], heads, 128, 1.2) or 256 % heads
    shares, length, planned = kernels.decode_wave_plan(lens, heads, 2048, 16, None, 128)
    assert planned is None or (shares, length) == (1, 0) and planned.tolist() == order.tolist()
    assert (shares, length) in ((1, 0), kernels.decode_share_plan(lens, heads, 2048, 16, None, 128))
    assert kernels.decode_wave_plan(lens[:511 // heads or 1], heads, 2048, 16, None, 128)[2] is None


@pytest.mark.parametrize("S,heads,tokens,window", [(64, 8, 500, None), (129, 4, 1000, None), (86, 6, 33, None), (64, 8, 3000, 1024)])
def test_sequences_of_one_length_are_not_sorted(monkeypatch, S, heads, tokens, window):
    """They meet their like in any order: the host, which eager and short steps wait for, plans nothing for them. A recorded
    step reads an order all the same."""
    from tie_amd import kernels

    monkeypatch.setattr(kernels, "whole_sequences_order", lambda *args: pytest.fail("sorted"))
    shares, length, order = kernels.decode_wave_plan([tokens] * S, heads, 4096, 16, window, 128)
    assert (shares, length) == (1, 0) and order.dtype.name == "int32" and order.tolist() == list(range(S))


def test_whole_sequences_in_order_where_shares_were_planned():
    """64 sequences of which the long ones come 32 apart: 1.9 times the mean as they come, 1.0 in order."""
    from tie_amd import kernels

    lens = [2000] * 8 + ([100] * 24 + [2000] * 8) + [100] * 24
    assert kernels.decode_share_plan(lens, 8, 2048, head_dim=128)[1] > 0
    assert kernels.decode_wave_plan(lens, 8, 2048, head_dim=128)[:2] == kernels.decode_share_plan(lens, 8, 2048, head_dim=128)
    lens = [2000] * 16 + [200] * 16 + [2000] * 16 + [200] * 16
    assert kernels.decode_share_plan(lens, 8, 2048, head_dim=128)[1] > 0
    shares, length, order = kernels.decode_wave_plan(lens, 8, 2048, head_dim=128)
    assert (shares, length) == (1, 0) and all(lens[a] + lens[b] == 2200 for a, b in zip(order[:32], order[32:]))


def test_shares_of_one_length_are_planned_for_sequences_of_very_different_lengths():
    import random

    from tie_amd import kernels

    rng = random.Random(0)
    assert kernels.decode_share_plan([2048] * 32, 8, 4096) == (kernels.decode_splits(32, 8, 4096), 0)
    assert kernels.decode_share_plan([4000, 3900, 4096] * 11, 8, 4096)[1] == 0          # about one length
    assert kernels.decode_share_plan([100, 4000], 8, 4096) == (kernels.decode_splits(2, 8, 4096), 0)   # many shares anyway
    assert kernels.decode_share_plan([32768] + [1024] * 7, 8, 32768) == (64, 21)          # one long sequence among short ones
    assert kernels.decode_share_plan([32768] * 8, 8, 32768)[1] == 0
    assert kernels.decode_share_plan([100, 4000] * 16, 8, 4096, block_size=8)[1] == 0     # the other kernel
    planned = 0
    for S, kvh, ctx in ((32, 8, 4096), (64, 8, 4096), (16, 8, 4096), (40, 4, 16384), (24, 8, 2048)):
        for i in range(20):
            lens = [rng.randint(20, ctx) for _ in range(S)] if i % 2 else [ctx] * 2 + [rng.randint(20, ctx // 6) for _ in range(S - 2)]
            shares, length = kernels.decode_share_plan(lens, kvh, ctx)
            equal = kernels.decode_splits(S, kvh, ctx)
            if length == 0:
                assert shares == equal
                continue
            tiles = [(n - 1) // 32 + 1 for n in lens]
            planned += 1
            assert shares >= equal and shares * length >= max(tiles) and length >= 4
            assert kvh * sum(-(-t // length) for t in tiles) <= (512 if S * kvh <= 128 else 768 if S * kvh <= 256 else 1024)
            before = -(-max(tiles) // equal)
            assert 2 * length <= before if equal <= 3 else 4 * length < before
    assert planned >= 20
    # a window bounds what a sequence shows: sequences far longer than the window are all of one length
    assert kernels.decode_share_plan([300, 4000] * 16, 8, 4096, window=256)[1] == 0
