"""Merge of split-K decode partials (decode_epilogue): split counts around the
merge's unroll and wave boundaries, both head sizes and every cache layout,
against the oracle; and a captured split decode replayed on changing inputs."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import assert_close, dev, memopt_C, to_dev

pytestmark = pytest.mark.gpu


def _case(seed, B, H, D, ctx):
    rng = np.random.default_rng(seed)
    M = (max(ctx) + 15) // 16
    nb = B * M + 1
    k = (rng.standard_normal((nb, 16, H, D)) * np.where(rng.random((nb, 16, H, D)) < 0.01, 8, 1)).astype(np.float16)
    v = rng.standard_normal((nb, 16, H, D)).astype(np.float16)
    q = rng.standard_normal((B, 1, H, D)).astype(np.float16)
    bt = rng.permutation(nb)[:B * M].reshape(B, M).astype(np.int32)
    return q, k, v, bt, np.array(ctx, np.int32)


@pytest.mark.parametrize("layout", ["pages", "rows", "fp16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("splits", [2, 3, 7, 24, 33, 64])
def test_split_counts_vs_oracle(layout, D, splits, monkeypatch):
    """ctx 0 (no split sees a key), 40 (most splits empty) and 1100."""
    monkeypatch.setenv("MEMOPT_DECODE_SPLITS", str(splits))
    q, k, v, bt, cl = _case(splits + D, 3, 2, D, [1100, 40, 0])
    kw = {}
    if layout == "fp16":
        kc, vc = to_dev(k), to_dev(v)
        want = O.paged_attention(q, k, v, bt, cl, 1100, 1100)
    elif layout == "pages":
        pages = O.to_int4_pages(k, v)
        kc = vc = to_dev(pages)
        want = O.paged_attention_int4(q, pages, bt, cl, 1100, 1100)
    else:
        (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
        kc, vc = to_dev(kq), to_dev(vq)
        kw = dict(key_scales=to_dev(ks), value_scales=to_dev(vs), kv_layout="token_major")
        want = O.paged_attention(q, O.dequantize_int4(kq, ks), O.dequantize_int4(vq, vs), bt, cl, 1100, 1100)
    got = memopt_C.dynamic_sparse_attention(to_dev(q), kc, vc, to_dev(bt), to_dev(cl), 1100, 1100, **kw)
    assert_close(got, want, what=f"{layout} decode in {splits} splits")


def test_captured_split_decode_replays():
    """A replay's counters start where the last replay of the same launch left
    them: every replay must merge its own splits, also after eager calls on
    the same workspace between replays."""
    q, k, v, bt, cl = _case(5, 1, 2, 128, [4096])
    pages = O.to_int4_pages(k, v)
    pg, dq = to_dev(pages), to_dev(q)
    call = memopt_C.PreparedAttention(dq, pg, pg, to_dev(bt), to_dev(cl), 4096, 4096)
    assert call.workspace_bytes > 0
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    g = torch.Generator(device=dev()).manual_seed(3)
    for i in range(6):
        dq.normal_(generator=g)
        want = call().clone()
        torch.cuda.synchronize()
        call.out.fill_(float("nan"))
        for _ in range(1 + i % 2):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(call.out, want)


@pytest.mark.parametrize("B,H", [(1, 1), (1, 8), (2, 12), (3, 5), (8, 3), (16, 6), (1, 40)])
def test_token_major_head_clusters(B, H):
    """Short calls (unclustered) over head counts and batches: every (sequence,
    head) is computed once, in its place."""
    rng = np.random.default_rng(B * 100 + H)
    ctx = [int(x) for x in rng.integers(1, 90, B)]
    q, k, v, bt, cl = _case(B + H, B, H, 64, ctx)
    (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
    want = O.paged_attention(q, O.dequantize_int4(kq, ks), O.dequantize_int4(vq, vs), bt, cl, 128, 128)
    got = memopt_C.dynamic_sparse_attention(to_dev(q), to_dev(kq), to_dev(vq), to_dev(bt), to_dev(cl), 128, 128,
                                            key_scales=to_dev(ks), value_scales=to_dev(vs), kv_layout="token_major")
    assert_close(got, want, what=f"{B} x {H} token-major heads")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,splits", [(1, 16, 1), (3, 32, 1), (2, 20, 2), (7, 8, 1), (8, 3, 1), (9, 12, 1),
                                        (5, 7, 3), (16, 40, 1), (1, 64, 8), (2, 1, 5), (12, 40, 1), (12, 10, 1),
                                        (11, 4, 6)])
def test_token_major_head_clusters_of_long_calls(B, H, splits, D, monkeypatch):
    """Calls whose block tables hold enough pages for head clusters (most of
    them unlinked here): fewer than 8 (sequence, split) units, 8, few and many
    between multiples of 8; cluster sizes 1 to 8, one to ten per unit."""
    monkeypatch.setenv("MEMOPT_DECODE_SPLITS", str(splits))
    rng = np.random.default_rng(B * 100 + H)
    ctx = [int(x) for x in rng.integers(1, 90, B)]
    q, k, v, bt, cl = _case(B + H, B, H, D, ctx)
    M = 6000 // (B * H) + 2
    wide = np.full((B, M), -1, np.int32)
    at = np.sort(rng.permutation(M)[:bt.shape[1]])     # pages spread over the table, so over the splits
    wide[:, at] = bt
    cl = np.array([16 * int(at[(c - 1) // 16]) + (c - 1) % 16 + 1 for c in ctx], np.int32)
    (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
    n = 16 * M
    want = O.paged_attention(q, O.dequantize_int4(kq, ks), O.dequantize_int4(vq, vs), wide, cl, n, n)
    got = memopt_C.dynamic_sparse_attention(to_dev(q), to_dev(kq), to_dev(vq), to_dev(wide), to_dev(cl), n, n,
                                            key_scales=to_dev(ks), value_scales=to_dev(vs), kv_layout="token_major")
    assert_close(got, want, what=f"{B} x {H} token-major heads of {D} in {splits} splits")
