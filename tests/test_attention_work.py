"""The host side of the block attention kernel: work items dealt to blocks."""
from types import SimpleNamespace

import pytest


def _batch(entries):
    cu = [0]
    for _, n in entries:
        cu.append(cu[-1] + n)
    return SimpleNamespace(host_cu_tokens=cu, host_start_pos=[p for p, _ in entries])


def _slices(P, n, G, c0, cols, window):
    ncols = n * G
    first, last = P + c0 // G, P + (min(c0 + cols, ncols) - 1) // G
    lo = max(0, first - window + 1) if window > 0 else 0
    return last // 32 - lo // 32 + 1


@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("bins", [1, 3, 32, 500])
def test_every_item_once_and_even_loads(bins, window):
    from tffinfer_amd.kernels.ops import _attention_block_work
    entries = [(0, 2048), (333, 200), (5, 1), (1000, 130), (0, 37)]
    G, cols = 4, 128
    batch = _batch(entries)
    items, starts, blocks, groups = _attention_block_work(batch, G, 8, window, "cpu", cols, bins=bins)
    assert groups in (1, 2)
    items, starts = items.tolist(), starts.tolist()
    want = sorted((r, c0) for r, (P, n) in enumerate(entries) for c0 in range(0, n * G, cols))
    assert sorted(map(tuple, items)) == want                      # no item lost, none twice
    assert blocks == len(starts) - 1 == min(bins, len(want))
    assert starts[0] == 0 and starts[-1] == len(items) and all(a < b for a, b in zip(starts, starts[1:]))
    loads = []
    for b in range(blocks):
        loads.append(sum(_slices(*entries[r], G, c0, cols, window) for r, c0 in items[starts[b]:starts[b + 1]]))
    biggest = max(_slices(*entries[r], G, c0, cols, window) for r, c0 in want)
    # longest-first dealing: no block carries more than the mean plus one item
    assert max(loads) <= sum(loads) / blocks + biggest
    if blocks == len(want):
        assert loads == sorted(loads, reverse=True)              # one item each, the longest first


def test_entry_filters():
    from tffinfer_amd.kernels.ops import _attention_block_work, _attention_work, _entries
    batch = _batch([(900, 1), (0, 300), (40, 1), (333, 150)])
    assert _entries(batch, "single") == [0, 2] and _entries(batch, "multi") == [1, 3]
    items, starts, blocks, _ = _attention_block_work(batch, 4, 2, 0, "cpu", 128, bins=64, which="multi")
    assert {r for r, _ in items.tolist()} == {1, 3}
    single = _attention_work(batch, 20, 16, "cpu", "single").tolist()     # 20 heads to a kv head: two tiles
    assert single == [[0, 0], [0, 16], [2, 0], [2, 16]]


def test_key_groups_and_blocks_follow_the_amount_of_work():
    """Little work: one block a CU, two groups of waves in it that share an item's slices; plenty:
    two blocks of one group a CU; large heads always one group, one block a CU."""
    from tffinfer_amd.kernels.ops import _attention_block_work
    short, long_ = _batch([(0, 2048)]), _batch([(0, 8192)])
    _, _, blocks, groups = _attention_block_work(short, 4, 8, 0, "cpu", num_cus=256)
    assert (blocks, groups) == (32, 2)
    _, _, blocks, groups = _attention_block_work(long_, 4, 8, 0, "cpu", num_cus=256)
    assert (blocks, groups) == (64, 1)
    _, _, blocks, groups = _attention_block_work(long_, 4, 8, 0, "cpu", num_cus=256, head_dim=256)
    assert (blocks, groups) == (32, 1)
    _, _, blocks, groups = _attention_block_work(long_, 4, 8, 0, "cpu", num_cus=256, key_groups=2)
    assert (blocks, groups) == (32, 2)
    # a portion of 2,048 tokens late in a long context is plenty of work as well
    _, _, blocks, groups = _attention_block_work(_batch([(6144, 2048)]), 4, 8, 0, "cpu", num_cus=256)
    assert (blocks, groups) == (64, 1)


def test_portions_take_the_blocks_that_end_first():
    """Short portions the blocks of eight waves, which begin and end sooner; longer ones those of four waves, with two key groups while
    there is no more than an item a block, with one where items of 256 columns spare a round; whatever the order of the portions."""
    from tffinfer_amd.kernels.ops import _prompt_blocks
    def pick(entries, G=4, nkv=8, window=0, d=128):
        return _prompt_blocks(_batch(entries), G, nkv, window, "cpu", "all", d, num_cus=256)
    assert [pick([(0, n)]) for n in (17, 96, 150, 333, 901, 2048, 6000, 32768)] == [0, 0, 0, 0, 2, 2, 1, 1]
    assert [pick([(0, n)], 32, 1, 0, 256) for n in (17, 96, 333, 6000)] == [0, 0, 1, 1]
    assert pick([(0, 901)], 5) == 2 and pick([(0, 333)], 1, 2) == 0
    mixed = [(0, 700), (2000, 300), (50, 20), (8000, 90)]
    assert pick(mixed, 4, 8, 1024) == pick(mixed[::-1], 4, 8, 1024) == 2 and pick(mixed) == 2
    assert pick([(9000, 500)]) == 2 and pick([(0, 40)] * 8) == 0
    assert pick([(0, 5), (100000, 40)] * 300) in (1, 2)      # more items than are dealt to find the longest block


@pytest.mark.parametrize("pool", [0, 16])
@pytest.mark.parametrize("window", [77, 0])
@pytest.mark.parametrize("entries", [[(0, 40), (3, 1), (900, 70)], [(0, 3001), (7, 1), (50, 1), (2000, 700), (0, 33)]])
def test_items_of_few_and_of_many_columns(entries, window, pool):
    """An item's slices are those of the keys its columns see, and of the blocks of keys before the window, whether the items are counted one
    by one or by arrays; the longest come first."""
    from tffinfer_amd.kernels.ops import _block_items
    for G, cols, which in ((4, 128, "all"), (5, 256, "multi")):
        want = []
        for r, (P, n) in enumerate(entries):
            for c0 in range(0, n * G, cols) if which == "all" or n > 1 else ():
                last = P + (min(c0 + cols, n * G) - 1) // G
                blocks = max(0, last - window + 1) // pool if pool and window else 0
                want.append((_slices(P, n, G, c0, cols, window) + -(-blocks // 32), r, c0))
        assert _block_items(_batch(entries), G, window, cols, which, pool if window else 0) == sorted(want, reverse=True)


def test_staged_tables_keep_shape_and_type_on_the_host():
    """The staging module's host form (what the work lists' tests above go through): every
    column comes back as a tensor of its own shape and element type, a copy of the array."""
    import numpy as np
    import torch
    from tffinfer_amd.kernels import staging
    a = np.arange(12, dtype=np.int32).reshape(-1, 2)
    b = np.asarray([0.5, 1.5, -2.0], dtype=np.float32)
    c = np.zeros((0, 2), dtype=np.int32)
    ta, tb, tc = staging.send("cpu", [a, b, c])
    assert ta.dtype == torch.int32 and tuple(ta.shape) == (6, 2) and ta.tolist() == a.tolist()
    assert tb.dtype == torch.float32 and tb.tolist() == b.tolist() and tuple(tc.shape) == (0, 2)
    a[0, 0] = 99
    assert ta[0, 0] == 0
