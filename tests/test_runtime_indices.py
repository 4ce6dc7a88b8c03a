"""Host-side index building of the paged cache: slots of page runs, batch
allocation and return of blocks (no kernel is launched)."""
import pytest


def _modules():
    import memopt_C
    from memopt_runtime import kv_cache
    return memopt_C, kv_cache


@pytest.mark.parametrize("start,count", [(0, 0), (0, 1), (15, 2), (5, 40), (47, 1)])
def test_slots_for(start, count):
    _, kv = _modules()
    pages = [7, 2, 9]
    want = [pages[p // 16] * 16 + p % 16 for p in range(start, start + count)]
    assert kv.slots_for(pages, start, count, 16) == want
    with pytest.raises(RuntimeError, match="position 16: logical block 1 is unlinked"):
        kv.slots_for([7, -1, 9], 3, 20, 16)


def test_slots_past_int32_raise(monkeypatch):
    """The last slot int32 holds, and the next one: an error, not a wrapped slot."""
    import torch
    _, kv = _modules()
    monkeypatch.setattr(kv.PagedKVCache, "device", torch.device("cpu"))
    cache = object.__new__(kv.PagedKVCache)
    cache.num_blocks = 2 ** 27 + 1
    cache.block_size, cache._pages, cache._len = 16, {0: [2 ** 27 - 1, 2 ** 27]}, {0: 0}
    assert cache.slot_mapping([0], 16)[-1] == 2 ** 31 - 1
    with pytest.raises(OverflowError, match="2147483648"):
        cache.slot_mapping([0], 17)


def test_batch_allocation_keeps_fifo_order():
    M, _ = _modules()
    M.reset_pool()
    with pytest.raises(RuntimeError, match="not initialized"):
        M.allocate_blocks(1)
    M._check(M._c_init_pool(6, 16, 1, 64, M.KV_INT4, 16, None, None, None))
    try:
        assert M.allocate_blocks(0) == [] and M.allocate_blocks(4) == [0, 1, 2, 3]
        assert M.allocate_blocks(3) is None and M.free_blocks_count() == 2   # all or none
        M.free_blocks([2, 0])
        with pytest.raises(RuntimeError, match="out of range"):
            M.free_blocks([1, 6])
        assert M.free_blocks_count() == 4                                     # nothing returned by the failed call
        assert [M.allocate_block() for _ in range(2)] == [4, 5] and M.allocate_blocks(2) == [2, 0]
    finally:
        M.reset_pool()
