"""The multi-query kernel without staging (csrc/direct.hip) against the CPU
oracle: INT4 pages, token-major codes with fp32 and fp16 scales, and fp16
pools, at the edges of its 16-query blocks, 32-token steps and splits."""
import numpy as np
import pytest
import torch

import oracle as O
from gpu_helpers import assert_close, dev, memopt_C, to_dev

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, D, bs, ctx, Lq, W, sinks, causal, unlink
    (1, 1, 64, 16, [2], 2, 64, 0, True, False),              # one partial chunk
    (2, 2, 128, 16, [17, 1], 2, 128, 4, True, False),         # ctx < q_len: a query that sees nothing
    (1, 2, 128, 16, [33], 15, 16, 2, True, False),            # odd chunk count, window inside one chunk
    (2, 3, 64, 16, [700, 63], 16, 100, 4, False, True),       # non-causal window and sinks, holes
    (1, 2, 128, 16, [1000], 17, 2048, 0, True, True),         # first size with two query blocks per wave
    (1, 2, 64, 16, [500], 33, 40, 70, True, False),           # sinks longer than the window, third block of 1 query
    (2, 2, 128, 48, [400, 96], 5, 512, 4, True, True),        # pages of three chunks (fp16, token-major)
    (1, 1, 128, 32, [2049], 7, 4096, 4, True, False),         # splits, last one partly empty
    (1, 2, 64, 16, [0], 3, 64, 4, False, False),              # empty context -> zeros
]


def _inputs(seed, B, H, D, bs, ctx, Lq, unlink):
    rng = np.random.default_rng(seed)
    M = max(1, (max(ctx) + bs - 1) // bs)
    nb = B * M + 2
    k = (rng.standard_normal((nb, bs, H, D)) * np.where(rng.random((nb, bs, H, D)) < 0.01, 8, 1)).astype(np.float16)
    v = rng.standard_normal((nb, bs, H, D)).astype(np.float16)
    q = rng.standard_normal((B, Lq, H, D)).astype(np.float16)
    bt = rng.permutation(nb)[:B * M].reshape(B, M).astype(np.int32)
    if unlink:
        bt[0, M // 2] = -1
        bt[-1, 0] = nb + 5
    return q, k, v, bt, np.array(ctx, np.int32)


@pytest.mark.parametrize("layout", ["pages", "rows", "rows_f16", "fp16"])
@pytest.mark.parametrize("case", CASES)
def test_direct_vs_oracle(case, layout):
    B, H, D, bs, ctx, Lq, W, sinks, causal, unlink = case
    if layout == "pages" and bs != 16:
        bs = 16
    q, k, v, bt, cl = _inputs(Lq * 7 + D, B, H, D, bs, ctx, Lq, unlink)
    kw, msl = {}, 1 << 20
    obt = np.where(bt >= k.shape[0], -1, bt).astype(np.int32)  # out-of-pool entries are skipped
    if layout == "fp16":
        kc, vc, kd, vd = to_dev(k), to_dev(v), k, v
    elif layout == "pages":
        pages = O.to_int4_pages(k, v)
        kc = vc = to_dev(pages)
        kd, vd = O.from_int4_pages(pages, D)
    else:
        (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
        if layout == "rows_f16":
            ks, vs = ks.astype(np.float16), vs.astype(np.float16)
        kc, vc = to_dev(kq), to_dev(vq)
        kw = dict(key_scales=to_dev(ks), value_scales=to_dev(vs), kv_layout="token_major")
        kd, vd = (O.dequantize_int4(c, s.astype(np.float32)) for c, s in ((kq, ks), (vq, vs)))
    want = O.paged_attention(q, kd, vd, obt, cl, msl, W, num_sink_tokens=sinks, causal=causal)
    got = memopt_C.dynamic_sparse_attention(to_dev(q), kc, vc, to_dev(bt), to_dev(cl), msl, W,
                                            num_sink_tokens=sinks, causal=causal, **kw)
    assert_close(got, want, what=f"{layout} {case}")
    # without a workspace the call runs unsplit
    one = memopt_C.PreparedAttention(to_dev(q), kc, vc, to_dev(bt), to_dev(cl), msl, W, num_sink_tokens=sinks,
                                     causal=causal, no_alloc=True, **kw)
    assert_close(one(), want, what=f"{layout} {case} no_alloc")


def test_direct_many_splits():
    """One (sequence, head) over 16400 tokens: 64 splits, in fp16 and both INT4 layouts."""
    for layout in ("pages", "rows", "fp16"):
        test_direct_vs_oracle((1, 1, 128, 16, [16400], 3, 1 << 20, 4, True, False), layout)
    torch.cuda.synchronize(dev())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [np.inf, np.nan, 3e4])
def test_direct_rows_non_finite_values(D, scale):
    """Token-major codes whose V scale is inf, NaN or large enough for fp16
    overflow in one group of one token: queries that do not see the token
    (causal, window) are as without it, the others get its inf or NaN in that
    group's dims only."""
    B, H, bs, n, Lq, W = 1, 2, 16, 200, 40, 30
    q, k, v, bt, cl = _inputs(3, B, H, D, bs, [n], Lq, False)
    (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
    key = n - 25                                     # seen by the queries at 175 .. 199 only
    page, G = int(bt[0, key // bs]), D // 64
    vs = vs.copy().reshape(-1, bs, H, G)
    vs[page, key % bs, 1, G - 1] = scale
    vs = vs.reshape(-1)
    got = memopt_C.dynamic_sparse_attention(to_dev(q), to_dev(kq), to_dev(vq), to_dev(bt), to_dev(cl), n, W,
                                            causal=True, key_scales=to_dev(ks), value_scales=to_dev(vs),
                                            kv_layout="token_major").float().cpu().numpy()
    with np.errstate(all="ignore"):
        kd = O.dequantize_int4(kq, ks)[bt[0]].reshape(-1, H, D)[:n].astype(np.float64)
        vd = O.dequantize_int4(vq, vs)[bt[0]].reshape(-1, H, D)[:n].astype(np.float64)
        for i in range(Lq):
            pos = n - Lq + i
            lo = max(0, pos - W + 1)
            for h in range(H):
                s = kd[lo:pos + 1, h] @ q[0, i, h].astype(np.float64) / D ** 0.5
                w = np.exp(s - s.max())
                want = ((w / w.sum())[:, None] * vd[lo:pos + 1, h]).sum(0).astype(np.float16).astype(np.float32)
                ok = np.isfinite(want)
                assert ok.all() == (pos < key or h == 0)
                assert_close(got[0, i, h][ok], want[ok], what=f"query {i} head {h}")
                np.testing.assert_array_equal(got[0, i, h][~ok], want[~ok])


@pytest.mark.parametrize("n", [200, 3000])                 # unsplit, and in splits
@pytest.mark.parametrize("D,scale", [(64, np.nan), (128, np.nan), (64, np.inf)])
def test_direct_rows_non_finite_scores(D, scale, n):
    """Token-major codes with a NaN or inf K scale (codes of both signs in the
    group, so the score is NaN), and a query holding a NaN: a query with such a
    score gives zeros, as the oracle states; all others are as without it."""
    B, H, bs, Lq, W, bad_q = 1, 2, 16, 40, 1 << 20, 3
    q, k, v, bt, cl = _inputs(5, B, H, D, bs, [n], Lq, False)
    (kq, ks), (vq, vs) = O.quantize_int4(k), O.quantize_int4(v)
    key = n - 25                                     # seen by the last 25 queries, head 1
    ks = ks.copy().reshape(-1, bs, H, D // 64)
    ks[int(bt[0, key // bs]), key % bs, 1, 0] = scale
    ks = ks.reshape(-1)
    q[0, bad_q, 0, 7] = np.nan
    args = (to_dev(q), to_dev(kq), to_dev(vq), to_dev(bt), to_dev(cl), n, W)
    kw = dict(causal=True, key_scales=to_dev(ks), value_scales=to_dev(vs), kv_layout="token_major")
    call = memopt_C.PreparedAttention(*args, **kw)
    assert (call.workspace_bytes > 0) == (n == 3000)
    got = call().cpu().numpy()
    with np.errstate(all="ignore"):
        want = O.paged_attention(q, O.dequantize_int4(kq, ks), O.dequantize_int4(vq, vs), bt, cl, n, W, causal=True)
    # (the oracle's additive mask lets the NaN key reach queries before it; they are as with a finite one)
    clean = O.paged_attention(q, O.dequantize_int4(kq, np.where(np.isfinite(ks), ks, 1).astype(ks.dtype)),
                              O.dequantize_int4(vq, vs), bt, cl, n, W, causal=True)
    hit = np.zeros((Lq, H), bool)
    hit[Lq - 25:, 1] = True
    hit[bad_q, 0] = True
    assert (got[0][hit] == 0).all() and (want[0][hit] == 0).all()
    assert_close(got[0][~hit], clean[0][~hit], what=f"queries without the score, n {n}")
    assert_close(memopt_C.PreparedAttention(*args, no_alloc=True, **kw)(), got, what="no_alloc")


@pytest.mark.parametrize("layout,B,H,D,n,Lq,W,causal,path", [
    ("pages", 4, 4, 128, 3540, 3540, 512, False, "staged"),
    ("fp16", 1, 32, 128, 1687, 1687, 512, True, "staged"),
    ("fp16", 16, 32, 64, 3568, 178, 1 << 20, True, "staged"),      # the blocks' repeated reads pass the caches
    ("pages", 1, 32, 128, 700, 700, 1 << 20, True, "direct"),
    ("pages", 4, 12, 64, 1000, 500, 1 << 20, True, "direct"),
    ("fp16", 2, 8, 128, 1024, 128, 1 << 20, False, "direct"),
])
def test_multi_query_path_by_estimate(layout, B, H, D, n, Lq, W, causal, path, multi_query_path):
    """Calls far to either side of the line between the direct kernel and the
    staged path run the faster one (equal bits), and both agree."""
    g = torch.Generator(device=dev()).manual_seed(Lq)
    nb = B * -(-n // 16)
    k, v = (torch.randn((nb, 16, H, D), generator=g, device=dev(), dtype=torch.float16) for _ in range(2))
    if layout == "pages":
        memopt_C.init_pool(nb, 16, H, D, kv_format="int4")
        memopt_C.write_cache(k.view(-1, H, D), v.view(-1, H, D), None,
                             torch.arange(nb * 16, dtype=torch.int32, device=dev()))
        k = v = memopt_C.get_int4_pages()
    q = torch.randn((B, Lq, H, D), generator=g, device=dev(), dtype=torch.float16)
    bt = torch.randperm(nb, generator=g, device=dev()).to(torch.int32).view(B, -1).contiguous()
    cl = torch.full((B,), n, dtype=torch.int32, device=dev())
    out = {}
    for name in ("auto", "staged", "direct"):
        multi_query_path(name)
        out[name] = memopt_C.dynamic_sparse_attention(q, k, v, bt, cl, n, W, causal=causal)
    assert torch.equal(out["auto"], out[path]) and not torch.equal(out["staged"], out["direct"])
    assert_close(out["direct"], out["staged"].cpu(), what="direct vs staged")


def test_more_query_blocks_than_a_grid_dimension():
    """2097152 queries (65536 blocks of 32, one more than the direct kernel's
    grid takes) with little work per query: served, as any other length."""
    B, H, D, n, Lq, W = 1, 1, 64, 40, 65536 * 32, 16
    q, k, v, bt, cl = _inputs(6, B, H, D, 16, [n], 2, False)
    rows = torch.randn(4096, D, generator=torch.Generator().manual_seed(6)).half()
    qd = rows.to(dev()).repeat(Lq // 4096, 1).reshape(B, Lq, H, D)
    got = memopt_C.dynamic_sparse_attention(qd, to_dev(k), to_dev(v), to_dev(bt), to_dev(cl), n, W)
    want = O.paged_attention(rows.numpy().reshape(1, 4096, 1, D), k, v, bt, cl, n, W)
    assert_close(got[:, :4096], want, what="first queries")
    same = got.reshape(Lq // 4096, 4096, D)
    assert all(torch.equal(same[i], same[0]) for i in range(0, Lq // 4096, 37)) and torch.equal(same[-1], same[0])
