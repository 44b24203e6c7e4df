"""Which steps a recording serves, and at which padded sizes: decided on the host, tested without a GPU."""
from types import SimpleNamespace

import pytest
import torch

from tlie_amd.engine.step import DecodeGraph, ModelRunner, PortionGraph, StepEntry


def runner():
    model = SimpleNamespace(device="cpu", spec=SimpleNamespace(vocab_size=100), graph_safe=True, dtype=torch.bfloat16)
    made = ModelRunner(model, cache=None)
    assert not made.use_graphs              # no recordings without a GPU
    made.use_graphs = True                  # (the decisions below do not touch the device)
    return made


def entries(counts, wants=None):
    wants = wants or [[count - 1] for count in counts]
    return [StepEntry(index, [1] * count, want) for index, (count, want) in enumerate(zip(counts, wants))]


def test_single_tokens_with_every_logit_wanted_replay_a_decode_recording():
    made = runner()
    assert made.replays(entries([1] * 5)) and made.replays(entries([1] * DecodeGraph.MAX_BATCH))
    assert not made.replays(entries([1] * (DecodeGraph.MAX_BATCH + 1)))
    assert not made.replays(entries([1, 2, 1])) and not made.replays(entries([1, 1], [[0], []]))
    assert [DecodeGraph.bucket_of(count) for count in (1, 2, 3, 9, 64, 65, 200)] == [1, 2, 4, 16, 64, 128, 256]


def test_portions_are_padded_to_the_recordings_sizes():
    made = runner()
    assert made.records(entries([5, 3])) == (16, 8)
    assert made.records(entries([16, 1])) == (32, 8)
    assert made.records(entries([33])) == (64, 8)
    assert made.records(entries([64, 1])) == (128, 8)
    assert made.records(entries([500, 12])) == (512, 8)
    assert made.records(entries([2] * 9)) == (32, 32)            # more than 8 sequences: up to 64, and no more than tokens
    assert made.records(entries([30] * 9)) == (320, 64)
    assert made.records(entries([1, 1], [[0], []])) == (16, 8)   # single tokens of which one is not wanted


def test_what_no_recording_serves():
    made = runner()
    assert made.records(entries([PortionGraph.MAX_TOKENS + 1])) is None
    assert made.records(entries([1] * (PortionGraph.MAX_SEQS + 1), [[] for _ in range(PortionGraph.MAX_SEQS + 1)])) is None
    assert made.records(entries([20], [list(range(20))])) is None               # more wanted rows than sequences
    assert made.records(entries([20, 20], [list(range(8)), [0]])) is None
    assert made.records(entries([20], [list(range(8))])) == (32, 8)
    assert made.records([StepEntry(0, [0], [0], source=3), StepEntry(1, [1, 2], [1])]) is None
    made.use_graphs = False
    assert made.records(entries([5, 3])) is None and not made.replays(entries([1]))


def prompt_step(tokens, before, seqs=1):
    import numpy as np
    return SimpleNamespace(max_new=tokens, num_seqs=seqs, num_tokens=tokens * seqs, max_context=before + tokens, scratch={}, tile_owner=None,
                           compute_units=256, tokens=torch.zeros(1),
                           host={"seq_start": np.arange(seqs + 1) * tokens, "seq_len": np.full(seqs, before + tokens)})


@pytest.mark.parametrize("head_dim", [96, 112, 128])
@pytest.mark.parametrize("tokens, before", [(64, 6000), (128, 4000), (512, 1500), (512, 7000), (1024, 5000), (2048, 0), (2048, 6000), (4096, 0)])
def test_the_variant_with_sinks_and_caps_takes_columns_that_fit_its_registers(tokens, before, head_dim):
    """Through LDS, 32 columns a wave of more than 96 dims spill 85 registers and more in the kernel's variant with a sink, chunks,
    capped scores or shared planes: it takes 16."""
    from tlie_amd import ops
    _, col_tiles, _, _, _, shared = ops.attention_plan(prompt_step(tokens, before), 4, 8, head_dim, extra=True)
    assert not shared or col_tiles == 1 or head_dim <= 96


@pytest.mark.parametrize("heads, kv_heads, dim, tokens, before, reach, extra, want", [
    # A window or chunk longer than the context is none: what the same step takes without it (or, in short contexts, no LDS)
    (16, 2, 128, 512, 6000, 8192, False, (2, 8, True)), (32, 8, 128, 1024, 5000, 8192, False, (2, 2, True)),
    (32, 8, 128, 64, 6000, 8192, True, (1, 8, True)), (16, 2, 128, 256, 600, 8192, True, (2, 1, False)),
    # One within the context bounds what is cut
    (32, 8, 128, 256, 3000, 1024, False, (2, 1, False)), (32, 8, 128, 64, 6000, 1024, True, (2, 4, False)), (32, 8, 128, 512, 6000, 1024, False, (1, 1, True)),
    (32, 8, 128, 2048, 6000, 1024, False, (2, 1, True)), (32, 8, 128, 2048, 6000, 1024, True, (1, 1, True)),
    # Heads of up to 32 dims keep their cut keys
    (16, 8, 32, 64, 6000, None, False, (1, 8, True)), (16, 8, 32, 256, 3000, None, True, (1, 2, True)), (32, 2, 16, 64, 6000, None, False, (1, 4, True)),
    # One and a half workgroups a unit of 96 dims are served by 16 columns a wave
    (24, 8, 96, 2048, 0, None, False, (1, 1, True)), (24, 8, 96, 2048, 0, None, True, (1, 1, True)),
    (24, 8, 96, 2048, 6000, None, True, (2, 1, True)), (32, 8, 80, 1536, 3000, None, True, (2, 1, True)), (24, 8, 96, 2048, 6000, None, False, (1, 1, True)),
    # Few tiles of their own keys: not cut
    (24, 8, 96, 256, 600, None, False, (2, 1, False)), (16, 2, 128, 64, 6000, None, False, (1, 8, True)),
])
def test_how_the_prompt_attention_is_cut_for_other_heads_and_reaches(heads, kv_heads, dim, tokens, before, reach, extra, want):
    """Calls that the lines drawn from 128 and 64 dims alone made up to five times slower: (columns a wave / 16, parts of the
    keys, through LDS) as measured for them."""
    from tlie_amd import ops
    _, col_tiles, nsplit, split_len, _, shared = ops.attention_plan(prompt_step(tokens, before), heads // kv_heads, kv_heads, dim, reach, extra)
    assert (col_tiles, nsplit, shared) == want
    if nsplit > 1:
        seen = before + tokens if reach is None else min(before + tokens, reach + 31 + 128 // (heads // kv_heads) + 1)
        assert split_len % 32 == 0 and nsplit * split_len >= seen


@pytest.mark.parametrize("batch, kv_heads, dim, context, parts", [
    (1, 8, 128, 8100, 29), (1, 8, 128, 16000, 32), (1, 8, 128, 5000, 16), (1, 4, 64, 5000, 16), (3, 4, 64, 16000, 16), (1, 4, 64, 16000, 32),
    (1, 8, 32, 16000, 16), (1, 8, 96, 8100, 29), (4, 2, 256, 8100, 29), (8, 2, 128, 16000, 16), (8, 4, 64, 2000, 8)])
def test_into_how_many_parts_a_decode_step_cuts_its_keys(batch, kv_heads, dim, context, parts):
    """More than 16 only for few tiles of many keys of large heads (elsewhere the merge takes longer than the parts give)."""
    from tlie_amd import ops
    _, _, nsplit, split_len, _, _ = ops.attention_plan(prompt_step(1, context - 1, batch), 4, kv_heads, dim)
    assert nsplit == parts and split_len % 32 == 0 and nsplit * split_len >= context


@pytest.mark.parametrize("counts, recorded, want", [
    ([512], False, True), ([7] * 60, False, False), ([8] * 60, False, True), ([400] + [1] * 8, False, True), ([400] + [1] * 9, False, False),
    ([2000] + [1] * 16, False, False), ([2048] + [1] * 16, False, True), ([1] * 300, False, False), ([300] + [0] * 7, True, True),
    ([300] + [0] * 63, True, False), ([1] * 64, True, False)])
def test_which_steps_bring_tokens_whose_slots_follow_one_another(counts, recorded, want):
    import numpy as np
    from tlie_amd import ops
    ctx = SimpleNamespace(max_new=max(counts), num_tokens=sum(counts), num_seqs=len(counts), tile_owner=object() if recorded else None,
                          host={"seq_start": np.concatenate([[0], np.cumsum(counts)])})
    assert ops.slots_follow(ctx) is want


@pytest.mark.parametrize("rows, outputs, inputs, gated, want", [
    (24, 22016, 4096, True, True), (16, 22016, 4096, True, True), (16, 11264, 2048, True, False), (17, 2048, 128, True, True), (64, 8192, 128, True, True),
    (64, 8193, 256, True, False), (32, 32768, 512, True, True), (32, 32769, 512, True, False), (64, 50000, 1024, False, False),
    (64, 50000, 1536, False, True), (4, 131072, 1024, False, False), (4, 32000, 2048, False, True), (64, 2048, 2048, False, False),
    (64, 1 << 10, (1 << 24) + 8, False, False)])
def test_which_products_keep_their_weights_in_a_ring(rows, outputs, inputs, gated, want):
    from tlie_amd import ops
    assert ops.ring_fits(rows, outputs, inputs, gated) is want
    if want:
        split_len, strips = ops.ring_plan(rows, outputs, inputs, 256, not gated)
        assert split_len % 64 == 0 and 1 <= strips <= 8 and (rows <= 48 or strips != 7) and (split_len >= inputs or not gated)


@pytest.mark.parametrize("counts, heads, kv_heads, dim, dtype, recorded, how, want", [
    # groups and sizes that the kernels know
    ([256], 32, 4, 64, "float32", False, {}, 1), ([255], 32, 4, 64, "float32", False, {}, 0), ([250, 1, 5], 32, 4, 64, "float32", False, {}, 2),
    ([4] * 64, 32, 4, 64, "float32", False, {}, 1), ([3] * 86, 32, 4, 64, "float32", False, {}, 0), ([256], 32, 4, 64, "bfloat16", False, {}, 1),
    ([256], 32, 4, 64, "float32", True, {}, 2), ([255], 32, 4, 64, "float32", True, {}, 0), ([1] * 300, 32, 4, 64, "float32", True, {}, 0),
    # sizes that they do not know, or no groups
    ([64], 32, 4, 64, "float32", False, dict(softcap=30.0), 1), ([63], 32, 4, 64, "float32", False, dict(softcap=30.0), 0),
    ([64], 32, 4, 64, "float32", False, dict(page_size=24), 1), ([64], 32, 4, 64, "float32", False, dict(page_size=8), 1),
    ([86], 32, 4, 32, "float32", False, dict(value_dim=48), 1), ([85], 32, 4, 32, "float32", False, dict(value_dim=48), 0),
    ([16], 32, 32, 64, "bfloat16", False, {}, 1), ([15], 32, 32, 64, "bfloat16", False, {}, 0), ([64], 32, 32, 64, "float32", False, {}, 1),
    ([7] * 64, 32, 32, 64, "float32", False, {}, 0), ([8] * 64, 32, 32, 64, "float32", False, {}, 1),
    ([86], 16, 2, 8, "bfloat16", False, {}, 1), ([85], 16, 2, 8, "bfloat16", False, {}, 0),
    # heads too large for it
    ([500], 32, 4, 65, "float32", False, {}, 0), ([500], 32, 4, 64, "float32", False, dict(value_dim=65), 0)])
def test_which_form_of_the_plain_attention_a_step_takes(counts, heads, kv_heads, dim, dtype, recorded, how, want):
    """0: a workgroup a token and head; 1: keys shared among a sequence's tokens; 2: both."""
    import numpy as np
    from tlie_amd import ops
    ctx = SimpleNamespace(num_tokens=sum(counts), max_new=max(counts), tile_owner=object() if recorded else None,
                          host={"seq_start": np.concatenate([[0], np.cumsum(counts)])})
    assert ops.attention_generic_plan(ctx, heads, kv_heads, dim, dtype=getattr(torch, dtype), **how) == want
    for group in (1, 3, 4, 16, 70):                           # pieces: equal ones of a sequence, as many columns as fit
        full = 64 // min(64, group)
        for tokens, seqs in ((1, 1), (100, 1), (60, 1), (128, 16), (1000, 64)):
            size = ops.generic_tile_tokens(tokens, seqs, group, 1)
            mean = -(-tokens // seqs)
            assert 1 <= size <= full and (mean > full or size == mean) and (mean <= full or 2 * size >= full or full == 1)


def test_the_skinny_products_launch_shape_is_one_the_kernel_takes():
    """Decided on the host from the sizes alone: every plan is within what the kernel takes, covers
    the inner size exactly, and for matrices that the policy balances the workgroups are no more
    than the compute units (one round) unless a round more is cheaper than more splits."""
    from tlie_amd import ops
    for rows in (1, 16, 17, 32, 33, 64):
        for out_features, in_features in ((2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (32000, 2048), (100, 520),
                                          (515, 1000), (64, 5632), (12288, 4096), (28672, 4096), (4096, 14336), (7, 8)):
            for units in (256, 304, 64):
                split_len, waves, strips = ops.skinny_plan(rows, out_features, in_features, units)
                assert split_len > 0 and split_len % 64 == 0 and 4 <= waves <= 16 and strips in (1, 2)
                assert strips == 1 or (rows > 32 and waves <= 8)
                nsplit = -(-in_features // split_len)
                assert (nsplit - 1) * split_len < in_features <= nsplit * split_len
                assert ops.skinny_plan(rows, out_features, in_features, units) == (split_len, waves, strips)    # (kept)
    # TinyLlama's four matrices at 64 rows on 256 compute units: one round of workgroups
    for out_features, in_features in ((2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632)):
        split_len, waves, strips = ops.skinny_plan(64, out_features, in_features, 256)
        workgroups = -(-out_features // (16 * waves * strips)) * -(-in_features // split_len)
        assert 128 < workgroups <= 256, (out_features, in_features, split_len, waves, strips)


def test_the_few_rows_products_launch_shape_is_one_the_kernel_takes():
    """Decided on the host from the sizes alone: waves 4, 8 or 16; an even number of rows of W a
    workgroup up to 16, or 32 with at most 8 waves; the gated product never an odd pairing."""
    from tlie_amd import ops
    for rows in (1, 2, 7, 8, 16):
        for out_features, in_features in ((2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (32000, 2048), (6144, 4096),
                                          (28672, 4096), (4096, 14336), (128256, 4096), (100, 520), (30, 64), (2112, 2048)):
            for epilogue in ("store", "rope", "silu", "residual"):
                for units in (256, 304, 64):
                    waves, rows_per_block = ops.gemm_rows_shape(out_features, in_features, epilogue, units, rows)
                    assert waves in (4, 8, 16)
                    assert (rows_per_block % 2 == 0 and 2 <= rows_per_block <= 16) or (rows_per_block == 32 and waves <= 8)
    assert ops.gemm_rows_shape(2560, 2048, "rope", 256, 8) == (16, 10)          # 256 workgroups, one a compute unit
    assert ops.gemm_rows_shape(2048, 2048, "residual", 256, 8) == (16, 16)      # a norm's sums follow: strips of 16
    assert ops.gemm_rows_shape(128256, 4096, "store", 256, 1) == (4, 16) and ops.gemm_rows_shape(128256, 4096, "store", 256, 8) == (4, 32)


def test_the_attention_work_list_equals_a_tile_by_tile_walk():
    """`ops.attention_tiles` makes a sequence's tiles at once; written out tile by tile here, the list must be
    the same rows in the same order (sequences in order, columns rising, then stably by keys seen, most first)."""
    import numpy as np
    from tlie_amd import ops

    def walk(seq_start, per_kv, col_tiles, seq_len):
        rows, keys = [], []
        for seq in range(len(seq_start) - 1):
            first, count = int(seq_start[seq]), int(seq_start[seq + 1] - seq_start[seq])
            for col0 in range(0, count * per_kv, 16 * col_tiles):
                rows.append((seq, first, count, col0))
                keys.append(int(seq_len[seq]) - count + min(count - 1, (col0 + 16 * col_tiles - 1) // per_kv) + 1 if seq_len is not None else 0)
        rows = np.asarray(rows, dtype=np.int32).reshape(-1, 4)
        if seq_len is not None and len(keys) > 1:
            rows = rows[np.argsort(-np.asarray(keys), kind="stable")]
        return rows
    rng = np.random.default_rng(3)
    for _ in range(100):
        counts = rng.integers(0, 90, rng.integers(1, 7))
        start = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
        lengths = (counts + rng.integers(0, 400, counts.shape[0])).astype(np.int32)
        per_kv, col_tiles = int(rng.choice([1, 3, 8, 32])), int(rng.choice([1, 2, 4, 8]))
        for seq_len in (None, lengths):
            made = ops.attention_tiles(start, per_kv, col_tiles, seq_len)
            assert made.dtype == np.int32 and made.flags["C_CONTIGUOUS"]
            assert np.array_equal(made, walk(start, per_kv, col_tiles, seq_len))


@pytest.mark.parametrize("heads, kv_heads, dim, tokens, before, want", [
    # (columns a wave / 16, parts of the keys, through LDS)
    (32, 8, 128, 2048, 0, (2, 1, True)), (32, 8, 128, 2048, 6000, (2, 1, True)), (32, 8, 128, 1536, 0, (1, 1, True)),
    (32, 8, 128, 1024, 2000, (1, 1, True)), (32, 8, 128, 1024, 5000, (2, 2, True)),
    (32, 8, 128, 512, 500, (1, 1, True)), (32, 8, 128, 512, 1500, (2, 4, True)),
    (32, 8, 128, 256, 500, (2, 1, False)), (32, 8, 128, 256, 1500, (1, 4, True)), (32, 8, 128, 256, 4000, (2, 8, True)),
    (32, 8, 128, 128, 700, (1, 4, True)),
    (32, 4, 64, 2048, 0, (1, 1, True)), (32, 4, 64, 512, 1500, (2, 1, False)), (32, 4, 64, 8192, 0, (2, 1, True)),
    (4, 2, 16, 1700, 0, (1, 1, True)),
])
def test_how_the_prompt_attention_is_cut(heads, kv_heads, dim, tokens, before, want):
    """The launch of the tiled attention kernel for one portion of `tokens` behind `before` positions on 256 compute units: parts
    cover the whole sequence in multiples of 32, and a window is never cut."""
    from types import SimpleNamespace
    import numpy as np
    import torch
    from tlie_amd import ops
    ctx = SimpleNamespace(max_new=tokens, num_seqs=1, num_tokens=tokens, max_context=before + tokens, scratch={}, tile_owner=None,
                          compute_units=256, tokens=torch.zeros(1), host={"seq_start": np.array([0, tokens]), "seq_len": np.array([before + tokens])})
    tiles, col_tiles, nsplit, split_len, waves, shared = ops.attention_plan(ctx, heads // kv_heads, kv_heads, dim)
    assert (col_tiles, nsplit, shared) == want
    assert tiles.shape[0] == -(-tokens * (heads // kv_heads) // (16 * col_tiles * (4 if shared else 1))) and (waves == 4 or not shared)
    if nsplit > 1:
        assert split_len % 32 == 0 and nsplit * split_len >= before + tokens > (nsplit - 1) * split_len
        assert ops.attention_plan(ctx, heads // kv_heads, kv_heads, dim, reach=1024)[2] == 1 or not shared
