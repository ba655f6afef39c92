"""The work list of decode attention (csrc/runtime.cpp, syn_decode_items): which sequence gets how
many of a step's workgroups.  No GPU: the list is laid out on the host."""
import random

import pytest

from synaptix_amd.kernels import runtime as rt

UNIT, MIN_UNITS = 32, 8


def _unpacked(lengths, n_splits, window=None):
    """(sequence, split, splits of the sequence, first) of every item; the length that an item carries and the
    table by sequence behind the items are checked here."""
    flat = rt.decode_items(lengths, n_splits, window)
    T, rows = len(lengths) * n_splits, len(lengths)
    assert len(flat) == 4 * T + 2 * rows
    out = []
    for at in range(T):
        seq, split_and_n, first, length = flat[4 * at:4 * at + 4]
        assert seq < 0 or length == lengths[seq]
        out.append((seq, split_and_n & 0xFFFF, split_and_n >> 16, first))
        if seq >= 0:
            assert flat[4 * T + 2 * seq:4 * T + 2 * seq + 2] == [first, split_and_n >> 16]   # the same by sequence
    return out


def _by_sequence(items):
    seqs = {}
    for at, (seq, split, n, first) in enumerate(items):
        if seq < 0:
            continue
        seqs.setdefault(seq, []).append((at, split, n, first))
    return seqs


def _check(lengths, n_splits, window=None):
    items = _unpacked(lengths, n_splits, window)
    assert len(items) == len(lengths) * n_splits
    seqs = _by_sequence(items)
    assert sorted(seqs) == list(range(len(lengths)))          # every sequence is there
    taken = set()
    for seq, rows in seqs.items():
        n = rows[0][2]
        assert [r[1] for r in rows] == list(range(n)) and all(r[2] == n for r in rows)   # each split once, in order
        first = rows[0][3]
        assert all(r[3] == first for r in rows) and first >= 0                           # one place for the sequence's partial results
        places = set(range(first, first + n))
        assert not (places & taken) and max(places) < len(items)
        taken |= places
        keys = lengths[seq] if window is None else min(lengths[seq], window)
        units = max(1, -(-keys // UNIT))
        assert n == 1 or units >= MIN_UNITS * n                                           # no split shorter than the least
    spare = [at for at, it in enumerate(items) if it[0] < 0]
    assert spare == list(range(len(items) - len(spare), len(items)))                      # spare items last
    return items, {s: rows[0][2] for s, rows in seqs.items()}


def test_sequences_of_one_length_get_equal_shares():
    _, n = _check([2060] * 8, 4)
    assert set(n.values()) == {4}
    _, n = _check([300] * 3, 5)      # 10 units: no second split of 8
    assert set(n.values()) == {1}


def test_longer_sequences_get_more_splits_and_lie_first():
    lengths = [64, 4000, 700, 3900, 1200, 90, 2500, 512]
    items, n = _check(lengths, 4)
    assert n[1] >= n[6] >= n[4] >= n[2] >= n[0] == 1
    assert sum(n.values()) <= 32 and n[1] > 4                 # what short sequences cannot use goes to long ones
    # in rounds: every sequence's first split, then the second of those that have one, ...; in a round the longest pieces first
    rounds = [sp for s, sp, _, _ in items if s >= 0]
    assert rounds == sorted(rounds)
    for r in set(rounds):
        pieces = [-(-(-(-lengths[s] // UNIT)) // k) for s, sp, k, _ in items if s >= 0 and sp == r]
        assert pieces == sorted(pieces, reverse=True)
    pieces = [-(-(-(-lengths[s] // UNIT)) // k) for s, sp, k, _ in items if s >= 0]
    # the longest piece of the uneven batch is shorter than with equal shares
    assert max(pieces) < -(-(-(-4000 // UNIT)) // 4)


def test_a_window_bounds_the_keys_that_count():
    _, n = _check([5000, 600], 4, window=512)
    assert n == {0: 2, 1: 2}                                  # both see 512 keys = 16 units: two splits of 8
    _, n = _check([5000, 600], 4)
    assert n[0] > n[1]


def test_padding_rows_and_random_batches_keep_the_list_whole():
    rnd = random.Random(3)
    for _ in range(200):
        rows = rnd.randint(1, 40)
        lengths = [rnd.choice([1, rnd.randint(1, 300), rnd.randint(1, 40000)]) for _ in range(rows)]
        _check(lengths, rnd.randint(1, 16), rnd.choice([None, None, 128, 4096]))


def test_refuses_an_empty_list():
    with pytest.raises(rt.CacheError):
        rt.decode_items([], 4)


def _binned(lengths, places, window=None):
    """The list of bins: every sequence's splits once each with places of their own for the partial results, the table
    behind the items, and the sum of units that every place gets."""
    T, rows = 2 * len(lengths), len(lengths)
    flat = rt.decode_bins(lengths, 2, places, window)
    assert len(flat) == 4 * T + 2 * rows
    seen, taken, load = {}, set(), [0] * places
    for at in range(T):
        seq, split_and_n, first, length = flat[4 * at:4 * at + 4]
        split, n = split_and_n & 0xFFFF, split_and_n >> 16
        if seq < 0:
            continue
        assert length == lengths[seq] and 0 <= split < n and flat[4 * T + 2 * seq:4 * T + 2 * seq + 2] == [first, n]
        assert (seq, split) not in seen and first + split not in taken and 0 <= first + split < T
        seen[(seq, split)] = n
        taken.add(first + split)
        units = -(-(lengths[seq] if window is None else min(lengths[seq], window)) // UNIT)
        load[at % places] += -(-units // n)
    n_of = {s: n for (s, _), n in seen.items()}
    assert sorted(n_of) == list(range(rows)) and len(seen) == sum(n_of.values())
    return load, n_of


@pytest.mark.parametrize("rows,places", [(33, 32), (64, 32), (65, 64), (96, 32), (128, 8), (257, 256)])
def test_bins_hold_every_piece_once_and_even_sums(rows, places):
    rnd = random.Random(rows)
    for window in (None, 500):
        for hi in (1, 40, 4000, 40000):
            lengths = [rnd.choice([1, rnd.randint(1, hi)]) for _ in range(rows)]
            load, n_of = _binned(lengths, places, window)
            units = [-(-(x if window is None else min(x, window)) // UNIT) for x in lengths]
            share = max(UNIT // 4, -(-sum(u for u in units if u > 1) // places))
            assert all(n == 1 for s, n in n_of.items() if units[s] <= share)       # only what is longer than a share is cut
            # every piece goes to the smallest sum: no sum is above their mean and the longest piece, over as many places as there are
            # pieces, or a half or a third as many
            flat = rt.decode_bins(lengths, 2, places, window)
            sums, longest, live = [0] * places, 0, 0
            for at in range(2 * rows):
                seq, split_and_n = flat[4 * at], flat[4 * at + 1] >> 16
                if seq >= 0 and units[seq] > 1:
                    piece = -(-units[seq] // split_and_n) + 4 + (2 if split_and_n > 1 else 0)      # what starting and merging it cost included
                    sums[at % places] += piece
                    longest, live = max(longest, piece), live + 1
            used = sum(x > 0 for x in sums)
            assert used >= min(places, -(-live // 3))
            assert not used or max(sums) <= sum(sums) / used + longest


def test_bins_pair_long_sequences_with_short_ones():
    lengths = [UNIT * (i + 1) for i in range(64)]                                  # 1 to 64 units
    load, n_of = _binned(lengths, 32)
    assert set(n_of.values()) == {1} and max(load) <= 1.05 * sum(load) / 32
    load, n_of = _binned([8000] + [500] * 63, 32)                                  # one alone is longer than five shares
    assert n_of[0] > 5 and max(load) <= 1.5 * sum(load) / 32
    load, _ = _binned([2048] * 33 + [1] * 31, 32)                                  # pairs in half of the places, not one pair among singles
    assert sum(u > 66 for u in load) == 16 and sum(64 <= u <= 66 for u in load) == 1


def test_bins_refuse_what_does_not_fit():
    for args in (([], 2, 8), ([5, 6], 2, 0), ([5] * 5, 1, 8)):
        with pytest.raises(rt.CacheError):
            rt.decode_bins(*args)


def test_bins_are_laid_out_for_layers_that_read_them():
    """Only the attention over one set of pages of plain heads reads a list; latent and window layers do not, nor a kernel that takes a
    kv head's queries in several workgroups, which the places do not count."""
    import torch
    from synaptix_amd.engine.graph import bin_places
    from synaptix_amd.parts import GqaAttention, KvNeed, NoPosition
    plain = lambda heads, kv, window=None: GqaAttention("a.", 64, heads, kv, 64, position=NoPosition(), window=window).cache_need()
    assert plain(32, 8) == KvNeed(8, 64) and hash(plain(32, 8)) == hash(plain(8, 8))      # layers of other heads share its pages
    needs = [plain(32, 8), plain(32, 8, 100), plain(128, 8), plain(256, 8), KvNeed(8, 64, 100, v_dim=64), KvNeed(1, 576, None, v_dim=512)]
    assert bin_places(33, needs, [0] * 6, torch.bfloat16) == [32, 32, 32, 0, 0, 0]
    assert bin_places(300, needs, [0] * 6, torch.bfloat16) == [32, 32, 32, 0, 0, 0]
    assert bin_places(32, needs, [0] * 6, torch.bfloat16) == [0] * 6                      # a workgroup a compute unit
    assert bin_places(33, needs, [2] + [0] * 5, torch.bfloat16)[0] == 0                   # every sequence is split
    assert bin_places(33, needs, [0] * 6, torch.float32) == [0] * 6


def test_only_lists_of_bins_are_merged_inside_large_launches():
    """A list that splits every sequence goes by the size of the grid, as a launch without a list does, also where more than 16 heads a
    kv head make it larger than sequences x kv heads."""
    from synaptix_amd.kernels import ops
    from synaptix_amd.kernels.build import load_library
    inside = load_library("attn_hd128").syn_attention_decode_merges_inside
    for rows, kv, heads in ((200, 1, 32), (100, 2, 64), (8, 8, 32), (32, 8, 32), (8, 8, 256), (30, 4, 128)):
        splits = ops.decode_splits(rows, kv, 512)
        assert splits > 1 or rows * kv >= 256
        chunks = -(-heads // kv // 16)
        assert bool(inside(rows, kv, heads, splits, 1)) == (rows * kv * chunks * splits <= 512) == bool(inside(rows, kv, heads, splits, 0))
    for rows, kv, heads in ((33, 8, 32), (64, 8, 32), (257, 1, 16)):
        assert ops.decode_splits(rows, kv, 512) == 1 and ops.decode_bins(rows, kv, heads // kv)
        assert inside(rows, kv, heads, ops.DECODE_BIN_SPLITS, 1)
