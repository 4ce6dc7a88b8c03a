"""autochunk_prefill where the pool cannot hold the whole prompt: the chunks
that fit are written and attended, then the call raises; and a shorter prompt
appended after them. Where there are fewer key rows than queries. And every
launch is made with the tensors' device current."""
import contextlib

import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import assert_close, dev, memopt_C

pytestmark = pytest.mark.gpu


def test_autochunk_out_of_pages():
    import memopt_runtime as R
    H, D, S, C = 2, 64, 400, 100
    q, k, v = (torch.randn(S, H, D, device=dev(), dtype=torch.float16) for _ in range(3))
    cache = R.PagedKVCache(14, H, D, kv_format="int4")        # 224 tokens: two chunks
    cache.add_sequence(0)
    with pytest.raises(RuntimeError, match="exhausted"):
        R.autochunk_prefill(cache, 0, q, k, v, window_size=64, chunk_tokens=C)
    assert cache.length(0) == 200 and len(cache.pages(0)) == 13 and memopt_C.free_blocks_count() == 1
    out = R.autochunk_prefill(cache, 0, q[200:220], k[200:220], v[200:220], window_size=64, chunk_tokens=7)
    kd, vd = O.from_int4_pages(memopt_C.get_int4_pages().cpu().numpy(), D)
    bt, ctx, n = R.attention_inputs(cache, [0])
    want = O.paged_attention(q[None, 200:220].cpu().numpy(), kd, vd, bt.cpu().numpy(), ctx.cpu().numpy(), n, 64,
                             causal=True)[0]
    assert n == 220
    assert_close(out, want, what="chunks of 7 after the failure")
    cache.free_sequence(0)
    assert memopt_C.free_blocks_count() == 14
    assert np.unique(memopt_C.allocate_blocks(14)).size == 14


@pytest.mark.parametrize("held,rows", [(0, 25), (30, 25), (30, 0), (0, 0)])
def test_autochunk_fewer_keys_than_queries(held, rows):
    """Queries past the last key row: each chunk writes the rows it has, and its
    queries end at the context written so far, as with append and an attention
    call per chunk."""
    import memopt_runtime as R
    H, D, S, C = 2, 64, 40, 10
    q, k, v = (torch.randn(S, H, D, device=dev(), dtype=torch.float16) for _ in range(3))
    cache = R.PagedKVCache(14, H, D, kv_format="int4")
    for s in (0, 1):
        cache.add_sequence(s)
        cache.append([s], k[None, :held], v[None, :held])
    out = R.autochunk_prefill(cache, 0, q, k[:rows], v[:rows], window_size=64, num_sink_tokens=4, chunk_tokens=C)
    assert cache.length(0) == held + rows
    for s0 in range(0, S, C):
        cache.append([1], k[None, s0:min(s0 + C, rows)], v[None, s0:min(s0 + C, rows)])
        bt, ctx, _ = R.attention_inputs(cache, [1])
        want = memopt_C.dynamic_sparse_attention(q[None, s0:s0 + C], *cache.key_value_pools(), bt, ctx,
                                                 held + s0 + C, 64, num_sink_tokens=4, causal=True)
        assert torch.equal(out[s0:s0 + C], want[0])
    assert len(cache.pages(0)) == len(cache.pages(1))


def test_autochunk_launches_on_the_tensors_device(monkeypatch):
    """The device guard (nothing to enter where the device is current already)
    is held around every launch, so a cache on another GPU than the current
    one launches there."""
    import memopt_C as M
    import memopt_runtime as R
    held, launches = [], []

    @contextlib.contextmanager
    def on(device):
        held.append(device)
        yield
        held.pop()

    def guarded(name):
        call = getattr(M, name)
        monkeypatch.setattr(M, name, lambda *a: (launches.append((name, list(held))), call(*a))[1])

    H, D, S = 2, 64, 50
    q, k, v = (torch.randn(S, H, D, device=dev(), dtype=torch.float16) for _ in range(3))
    cache = R.PagedKVCache(8, H, D, kv_format="int4")
    cache.add_sequence(0)
    monkeypatch.setattr(M, "_on", on)
    guarded("_c_attn")
    guarded("_c_write")
    R.autochunk_prefill(cache, 0, q, k, v, chunk_tokens=20)
    assert [n for n, _ in launches] == ["_c_write", "_c_attn"] * 3
    assert all(devices[-1:] == [q.device] for _, devices in launches)
