"""autochunk_prefill where the pool cannot hold the whole prompt: the chunks
that fit are written and attended, then the call raises; and a shorter prompt
appended after them."""
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
