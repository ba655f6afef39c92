"""The native host runtime on its own: the integer tables of a step, written from the cache's state."""
import ctypes as C

import numpy as np
import pytest
import torch

from synaptix_amd.cache import SequenceCache, CacheError
from synaptix_amd.engine.batch import StepContext, StepLayout, fill_host_buffer
from synaptix_amd.kernels import runtime as rt
from synaptix_amd.parts.base import KvNeed


def make_cache():
    return SequenceCache([KvNeed(2, 16), KvNeed(1, 32, window=100)], 64 * 12, 4, torch.float32, "cpu")


def test_layout_puts_the_arrays_one_after_another():
    lay = StepLayout(7, 2, 3, [4, 2])
    assert lay.off == {"tokens": (0, 7), "tok_seq": (7, 7), "tok_pos": (14, 7), "seq_start": (21, 3),
                       "seq_past": (24, 2), "seq_len": (26, 2), "seq_slot": (28, 2), "want": (30, 3)}
    assert lay.table_off == [(33, 8), (41, 4)] and lay.total == 45
    assert StepLayout(0, 0, 0, []).total == 1


def test_step_tables_follow_the_cache():
    c = make_cache()
    a, b = c.acquire(), c.acquire()
    c.reserve(a, 70), c.commit(a, 70)
    c.reserve_step([b, a], [3, 2])
    lay = StepLayout(5, 2, 2, [c.table_width(g, [b, a]) for g in range(2)])
    assert lay.widths == [2, 2]
    host = np.full(lay.total + 3, -7, dtype=np.int32)
    fill_host_buffer(lay, host, c, [b, a], np.array([11, 12, 13, 21, 22]), [3, 2], [2, 4])

    def arr(name):
        o, n = lay.off[name]
        return host[o:o + n].tolist()

    assert arr("tokens") == [11, 12, 13, 21, 22]
    assert arr("tok_seq") == [0, 0, 0, 1, 1]
    assert arr("tok_pos") == [0, 1, 2, 70, 71]
    assert arr("seq_start") == [0, 3, 5] and arr("seq_past") == [0, 70] and arr("seq_len") == [3, 72]
    assert arr("seq_slot") == [b, a] and arr("want") == [2, 4]
    for g in range(2):
        o, n = lay.table_off[g]
        assert host[o:o + n].reshape(2, 2).tolist() == c.page_table(g, [b, a], width=2).tolist()
    assert host[lay.total:].tolist() == [-7, -7, -7]            # nothing written behind the tables
    with pytest.raises(CacheError, match="not live"):
        fill_host_buffer(lay, host, c, [b, 3], np.zeros(5), [3, 2], [2, 4])
    with pytest.raises(ValueError):
        fill_host_buffer(lay, host[:10], c, [b, a], np.zeros(5), [3, 2], [2, 4])


def test_decode_tables_pad_with_a_spare_page():
    c = make_cache()
    a, b = c.acquire(), c.acquire()
    c.reserve(a, 130), c.commit(a, 130)
    c.reserve(b, 5), c.commit(b, 5)
    c.reserve(a, 1), c.reserve(b, 1)
    rows, widths, spare = 4, [4, 4], [12, 12]
    lay = StepLayout(rows, rows, rows, widths)
    item_splits = [0, 3]                       # the second group keeps a work list for its attention: 4 x 3 items
    host = np.zeros(lay.total + 2 * rows + 4 * rows * 3 + 2 * rows, dtype=np.int32)
    temps, unis = (C.c_float * 2)(0.5, 0.0), (C.c_float * 2)(0.25, 0.75)
    rt.check(rt.lib().syn_decode_fill(c._h, rows, 2, rt.ints([a, b]), rt.ints([9, 8]), 2, rt.ints(widths),
                                      rt.ints(spare), temps, unis, rt.ints(item_splits), host.ctypes.data))

    def arr(name):
        o, n = lay.off[name]
        return host[o:o + n].tolist()

    assert arr("tokens") == [9, 8, 0, 0] and arr("tok_pos") == [130, 5, 0, 0]
    assert arr("tok_seq") == [0, 1, 2, 3] and arr("seq_start") == [0, 1, 2, 3, 4]
    assert arr("seq_past") == [130, 5, 0, 0] and arr("seq_len") == [131, 6, 1, 1]
    assert arr("seq_slot") == [a, b, -1, -1] and arr("want") == [0, 1, 2, 3]
    full = host[lay.table_off[0][0]:][:16].reshape(4, 4)
    own = c.page_table(0, [a, b], width=4)
    assert full[0, :3].tolist() == own[0, :3].tolist() and full[1, 0] == own[1, 0]
    assert full[0, 3] == 12 and full[1, 1:].tolist() == [12, 12, 12] and (full[2:] == 12).all()
    f = host[lay.total:lay.total + 2 * rows].view(np.float32)
    assert f.tolist() == [0.5, 0.0, 0.0, 0.0, 0.25, 0.75, 0.0, 0.0]
    flat = host[lay.total + 2 * rows:].tolist()
    assert flat == rt.decode_items([131, 6, 1, 1], 3)                          # from the lengths that the step has
    items = [flat[4 * i:4 * i + 4] for i in range(12)]
    assert sorted(i[0] for i in items[:4]) == [0, 1, 2, 3] and all(i[0] == -1 for i in items[4:])   # too short to split
    assert all(i[1] == 1 << 16 for i in items[:4]) and sorted(i[3] for i in items[:4]) == [1, 1, 6, 131]
    assert flat[48:] == [x for i in range(4) for x in (next(it[2] for it in items if it[0] == i), 1)]   # the same by sequence
    with pytest.raises(CacheError, match="width"):
        rt.check(rt.lib().syn_decode_fill(c._h, rows, 2, rt.ints([a, b]), rt.ints([9, 8]), 2, rt.ints([2, 4]),
                                          rt.ints(spare), None, None, None, host.ctypes.data))
    with pytest.raises(CacheError, match="rows"):
        rt.check(rt.lib().syn_decode_fill(c._h, 1, 2, rt.ints([a, b]), rt.ints([9, 8]), 2, rt.ints(widths),
                                          rt.ints(spare), None, None, None, host.ctypes.data))


def test_sums_of_short_prompts_stay_in_32_bits_whatever_the_number_of_slices():
    """q, k and v of prompts whose product fills at most half of the compute units reach their norm as 32-bit sums, also at the
    sizes where one slice of K is the fastest: the number of slices decides the speed, not the precision."""
    import torch
    from synaptix_amd.kernels import ops
    from synaptix_amd.parts.linear import Matrix, keeps_sums, product_slices
    one = 0
    for N, K, tokens in ((6144, 2560, (258, 320, 540, 640, 961, 1280)), (4096, 2048, (713, 1024, 1153, 1408, 1537, 2048)),
                         (3072, 1024 * 2, (321, 2560)), (6144, 4096, (66, 129, 250, 300, 700, 1280)), (10240, 5120, (256, 700))):
        w = Matrix(torch.zeros((N, K), dtype=torch.bfloat16), keep_rows=True)
        for M in tokens:
            assert ops.gemm_keeps_sums(M, N, K, torch.bfloat16) and keeps_sums(M, w, torch.bfloat16), (M, N, K)
            one += product_slices(M, w, torch.bfloat16) == 1
    assert one          # (sizes of one slice were among them)
    for M in (2048, 5000):
        assert not ops.gemm_keeps_sums(M, 6144, 4096, torch.bfloat16)
    for M in (1, 64, 300, 5000):
        for N, K in ((6144, 4096), (64, 64), (4096, 2052), (30000, 4096)):
            assert not ops.gemm_keeps_sums(M, N, K, torch.float32)
            assert ops.gemm_keeps_sums(M, N, K, torch.bfloat16) >= (ops.gemm_slices(M, N, K, torch.bfloat16) > 1)


def test_sums_that_were_handed_on_in_32_bits_stay_so_whatever_the_fit_of_the_tiles_says():
    """Rows of wider and longer products whose q, k and v have reached their norm as 32-bit sums, and 65 to 128 rows of short ones: what
    picks tiles and slices may change, none of these may come to be rounded."""
    import torch
    from synaptix_amd.kernels import ops
    kept = {(10240, 5120): [(1537, 1792)], (12288, 5120): [(1281, 1536)], (7168, 5120): [(2305, 2560)], (16384, 4096): [(1025, 1152)],
            (10240, 8192): [(1537, 1920), (2049, 2112), (3649, 4096), (4865, 5376)],
            (8192, 8192): [(1025, 1152), (2049, 2304), (2817, 2880), (4609, 5120), (6145, 6656)], (8192, 4096): [(2113, 2304)],
            (5120, 5120): [(3073, 3648), (4801, 4864)], (4096, 4096): [(4417, 4608)], (16384, 8192): [(1281, 1344), (2305, 2560), (3073, 3264)],
            (3072, 1024): [(65, 128)], (6144, 1536): [(65, 128)], (512, 1024): [(65, 128)]}
    for (N, K), ranges in kept.items():
        for lo, hi in ranges:
            for M in (*range(lo, hi, 7), hi):
                assert ops.gemm_keeps_sums(M, N, K, torch.bfloat16), (M, N, K)
    # rounded as before: prompts of the 8B and 4B shapes beyond half of the compute units, short products of more rows, small ones
    for M, N, K in ((1281, 6144, 4096), (2048, 6144, 4096), (2600, 6144, 4096), (1281, 6144, 2560), (4096, 6144, 2560), (129, 3072, 1024),
                    (2048, 3072, 1024), (100, 256, 1024), (2048, 10240, 5120)):
        assert not ops.gemm_keeps_sums(M, N, K, torch.bfloat16), (M, N, K)


def test_host_side_rules_of_the_kernels_stay_within_their_kernels_limits():
    """The numbers of splits and slices that the host picks: pure functions, checked over a grid of sizes."""
    import torch
    from synaptix_amd.kernels import ops
    for n_seqs in (1, 2, 3, 8, 17, 64, 300):
        for n_kv in (1, 2, 8):
            for pages in (1, 2, 8, 9, 33, 96, 128, 512, 4096):
                s = ops.decode_splits(n_seqs, n_kv, pages)
                assert 1 <= s <= 64 and s <= pages
                assert s == 1 or pages // s >= 4          # a split keeps at least four blocks
    assert ops.decode_splits(64, 8, 33) == 1 and ops.decode_splits(1, 8, 33) > 1
    for M in (1, 8, 9, 32, 33, 64, 65, 128, 512, 2048, 8192):
        for N, K in ((4096, 4096), (6144, 4096), (4096, 12288), (151936, 4096), (64, 64), (4096, 1000)):
            s = ops.gemm_slices(M, N, K, torch.bfloat16)
            assert 1 <= s <= 8
            if s > 1:
                step = ((K + s - 1) // s + 127) // 128 * 128
                assert (s - 1) * step < K, "no slice may be empty"
                assert K % 8 == 0 and (M <= 64 or K % 128 == 0)
            assert ops.gemm_slices(M, N, K, torch.float32) == 1


def test_cut_products_take_the_tiles_whose_slices_fill_the_compute_units():
    """57 to 64 and 177 to 256 rows: slices of the tiles that load straight into LDS where these fill the compute units (a power of two), of the
    streamed tiles elsewhere."""
    import torch
    from synaptix_amd.kernels import ops
    cut = lambda M, N, K: ops.gemm_slices(M, N, K, torch.bfloat16)
    for N, K, s in ((6144, 4096, 4), (4096, 4096, 8), (4096, 12288, 8), (6144, 2560, 4), (2560, 4096, 8), (2560, 9728, 8), (4096, 2048, 4), (2048, 2048, 4),
                    (2048, 8192, 8), (8192, 28672, 4), (3072, 1024 * 3, 4)):
        assert {cut(M, N, K) for M in (33, 48, 56, 57, 60, 64)} == {s}, (N, K)
    for N, K, few, s in ((10240, 5120, 2, 3), (5120, 8192, 4, 6), (5120, 25600, 4, 6)):
        assert cut(56, N, K) == few and {cut(M, N, K) for M in (57, 64)} == {s}, (N, K)
    for N, K, s in ((6144, 4096, 2), (4096, 12288, 4), (6144, 6144, 2), (7168, 5120, 2), (3072, 8192, 4)):
        assert {cut(M, N, K) for M in (177, 224, 256)} == {s}, (N, K)


def test_cut_products_over_plain_rows_keep_the_slices_that_fill_the_compute_units():
    """W in plain rows, which the streamed tiles read in short pieces: powers of two up to 128 rows whatever W, above where they fill."""
    import torch
    from synaptix_amd.kernels import ops
    cut = lambda M, N, K: ops.gemm_slices(M, N, K, torch.bfloat16, packed=False)
    for N, K, s in ((6144, 2560, 4), (4096, 4096, 8), (2560, 9728, 8), (10240, 5120, 2), (5120, 8192, 4), (4096, 12288, 8)):
        assert {cut(M, N, K) for M in (48, 57, 64, 65, 96, 128)} == {s}, (N, K)
    for N, K, s in ((4096, 4096, 4), (8192, 4096, 2), (6144, 4096, 2), (4096, 12288, 4)):
        assert {cut(M, N, K) for M in (177, 256)} == {s}, (N, K)


def test_experts_weights_are_loaded_past_the_caches_where_most_segments_are_one_tile():
    """Non-temporal loads of W were faster for up to 224 rows an expert on average, and slower beyond, where several tiles of rows read it."""
    from synaptix_amd.kernels.build import load_library
    once = load_library("core").syn_grouped_stream_once
    assert all(once(r) for r in (48, 100, 188, 224)) and not any(once(r) for r in (225, 256, 310, 750, 1024, 2048))


def test_experts_tiles_hold_the_rows_of_a_segment():
    """Tiles of 64 rows took up to twice as long as the others with 80 and 100 rows an expert, tiles of 128 up to twice with 160 and more."""
    from synaptix_amd.kernels.build import load_library
    rows = load_library("core").syn_grouped_stream_rows
    assert {rows(r) for r in (48, 64, 80)} == {128} and {rows(r) for r in (81, 128, 188, 310, 2048)} == {256}


def test_32_bit_prompts_share_workgroups_only_where_that_was_measured_to_pay():
    """Steps timed with a wave a row and with 16 rows a workgroup: the latter walks a workgroup's sequences one after another, which single
    tokens behind long contexts beside a prompt make up to six times slower than the former, and many short prompts half as slow again."""
    from synaptix_amd.kernels import ops
    pays = lambda past, new, *heads: ops.prompt_rows_pay(past, new, *heads)
    for nh, nkv, hd in ((32, 8, 128), (32, 32, 128), (12, 12, 96), (32, 32, 64)):
        assert pays([0] * 3, [120, 137, 233], nh, nkv, hd) and pays([0], [600], nh, nkv, hd) and pays([700] * 2, [260] * 2, nh, nkv, hd)
    for nh, nkv, hd in ((32, 32, 128), (12, 12, 96), (8, 8, 64), (32, 32, 64)):
        assert not pays([0] + [1500] * 20, [400] + [1] * 20, nh, nkv, hd)
        assert not pays([0] * 6 + [2000] * 10, [64] * 6 + [1] * 10, nh, nkv, hd)
    assert not pays([0] + [2000] * 3, [100] + [1] * 3, 32, 8, 128) and not pays([2000] * 3 + [0], [1] * 3 + [100], 40, 8, 80)
    for n, each in ((2, 33), (8, 17), (8, 33), (16, 17)):
        assert not pays([0] * n, [each] * n, 32, 8, 128)
    assert pays([0] * 4, [64] * 4, 32, 8, 128) and pays([100] * 8, [17] * 8, 32, 8, 128) and pays([300] * 64, [16] * 64, 32, 8, 128)
    assert not pays([0], [60], 32, 8, 128) and not pays([5000] * 70, [1] * 70, 32, 8, 128)
    layout = StepLayout(57 + 60, 2, 0, [1])
    ctx = StepContext(layout, torch.zeros(layout.total, dtype=torch.int32), torch.float32, [0, 1], [700, 0], [57, 60], None)
    assert ctx.prompt_rows_pay(32, 8, 128) and not ctx.prompt_rows_pay(4, 4, 16)


def test_a_routers_product_runs_in_slices_only_where_that_was_measured_to_pay():
    from synaptix_amd.parts.feedforward import router_slices_pay
    for tokens, experts in ((1500, 48), (1500, 128), (1500, 256), (40, 256), (16, 48), (16, 128), (8, 8), (8, 128)):
        assert router_slices_pay(tokens, experts), (tokens, experts)
    for tokens, experts in ((1, 8), (1, 256), (8, 256), (16, 256), (17, 256), (16, 1024), (100, 1024), (1500, 1024), (4000, 1024)):
        assert not router_slices_pay(tokens, experts), (tokens, experts)


def test_keys_and_values_of_latent_prompts_stay_within_their_memory():
    """Whatever the step: what the heads' keys and values take at a time, with the rows that they are made from, is no more than the limit
    or the queries and results in the latent's space that the step does without, down to one head; every head is computed; steps below the limit go in one piece."""
    from synaptix_amd.kernels import ops
    for heads in (1, 2, 3, 8, 32, 128):
        for rank in (128, 512):
            for tokens in (129, 1500, 8000, 16000, 60000):
                for ratio in (1, 3, 8):
                    rows = tokens * ratio // 64 * 64
                    k = ops.latent_expanded_heads(rows, tokens, heads, rank, 64)
                    assert 1 <= k <= heads
                    taken = 512 * rows * k + 2 * rows * (rank + 64)
                    assert k == 1 or taken <= max(ops.LATENT_EXPANDED_BYTES, 4 * tokens * heads * rank), (heads, rank, tokens, ratio, k)
                    assert k == heads or 512 * rows * heads + 2 * rows * (rank + 64) > ops.LATENT_EXPANDED_BYTES
    assert ops.latent_expanded_heads(128000, 16000, 32, 512, 64) == 11 and ops.latent_expanded_heads(15232, 7000, 32, 512, 64) == 32
