"""A6 workspace sizes, host side (CPU only; no kernel is launched)."""

from __future__ import annotations

import random

import pytest

from nanoengine_amd import _native


@pytest.fixture(scope="module")
def size():
    if not _native.library_path().exists():
        pytest.skip("libnanoengine_hip.so is not built (run __graft_entry__.build())")
    return _native.load().ne_paged_attention_workspace_size


# (sequences, max_q_len, max_ctx_len): a chunk of a long prompt beside short prompts, one long
# sequence in a graph's 64 slots of 17 rows, one in 256 slots
@pytest.mark.parametrize("seqs,q,ctx", [(13, 300, 16000), (64, 17, 16384), (256, 20, 4096)])
def test_a_long_context_among_many_sequences_can_be_split(size, seqs, q, ctx):
    """Prefill splits follow the sequences' lengths, which only the device knows: the partials
    have room for one long sequence's splits (8 heads x 16 parts of 64 rows, 130 floats each)
    however many others the bounds allow."""
    assert size(seqs, 16, 8, q, ctx, 0) >= 8 * 16 * 64 * 130 * 4


def test_the_split_rule_needs_no_more_parts_than_there_is_room_for():
    """A tile of n >= 1.5 S stages in round(n / S) parts, S = max(ceil(T heads / 256), least):
    at most 341 parts of all heads, 256 beside the tiles' first ones, and no part without a
    stage, whatever the lengths."""
    rng = random.Random(0)
    for _ in range(3000):
        heads, least, longest = rng.choice([1, 2, 3, 8, 16]), rng.choice([2, 4]), rng.choice([3, 9, 100, 3000])
        stages = [rng.randint(0, longest) if rng.random() < 0.3 else rng.randint(0, 3) for _ in range(rng.randint(1, 300))]
        share = max(-(-sum(stages) * heads // 256), least)
        parts = {i: (n + share // 2) // share for i, n in enumerate(stages) if 2 * n >= 3 * share}
        assert all(2 <= k <= (stages[i] + 1) // 2 for i, k in parts.items())
        assert heads * sum(parts.values()) <= 341
        assert heads * sum(k - 1 for k in parts.values()) <= 256
        assert heads * len(parts) <= 341 // 2


# (8, 2,048, 4,096): a prefill chunk whose engine verifies 8 sequences of 5 rows in the same
# buffer; (64, 17, 4,096): 16 guesses, and fewer
@pytest.mark.parametrize("heads", [(16, 8), (8, 8), (24, 2), (40, 1)])
@pytest.mark.parametrize("largest", [(8, 2048, 4096), (64, 17, 4096), (64, 895, 895), (1, 8192, 16384), (256, 300, 300)])
def test_a_buffer_for_the_largest_shape_holds_every_smaller_one(size, heads, largest):
    rng = random.Random(sum(largest))
    bound = size(largest[0], *heads, *largest[1:], 0)
    for _ in range(4000):
        seqs, q, ctx = (max(1, min(n, int(n * 2 ** -rng.uniform(0, 12)))) for n in largest)
        assert size(seqs, *heads, q, ctx, 0) <= bound, (seqs, q, ctx)
