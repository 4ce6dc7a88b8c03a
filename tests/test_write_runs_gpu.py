"""write_cache into INT4 pages when pages start at any token of a 16-token
group: runs of pages between heads and tails that scatter, bytes against the
oracle."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import memopt_C, same_bits, special_fp16, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", [
    [5, 16, 40],            # page 2 starts at token 5 of the first group
    [31, 33, 1, 47],        # starts at tokens 15 and 0 of a group, tails of 15 and 1
    [1] * 15 + [64],        # scattered tokens, then pages from token 15 on
    [16, 15, 16, 17, 100],
    [200],
    [5, 16, 40, 31, 1] + [997] * 8,  # enough elements for pages from any token (1.5 M at D = 64)
    [997] * 7 + [833],               # just too few
])
def test_write_page_runs(D, lens):
    """Sequences back to back, each at the start of its own pages (permuted);
    one sequence's second page is replaced by scattered slots, and one slot
    lies past the pool (skipped: its group is no page)."""
    rng = np.random.default_rng(sum(lens) + D)
    H, bs = 3, 16
    pages = [int(np.ceil(n / bs)) for n in lens]
    nb = sum(pages) + 3
    perm = rng.permutation(nb)
    slots, at = [], 0
    for n, m in zip(lens, pages):
        p = perm[at:at + m]
        at += m
        s = p[np.arange(n) // bs] * bs + np.arange(n) % bs
        if m > 3:
            s[bs:2 * bs] = s[bs:2 * bs][rng.permutation(bs)]
            s[3 * bs] = nb * bs + 7
        slots.append(s)
    slots = np.concatenate(slots).astype(np.int32)
    T = slots.size
    k = special_fp16((T, H, D), 1) if T * H * D >= 512 else rng.standard_normal((T, H, D)).astype(np.float16)
    v = rng.standard_normal((T, H, D)).astype(np.float16)
    memopt_C.init_pool(nb, bs, H, D, kv_format="int4")
    memopt_C.write_cache(to_dev(k), to_dev(v), to_dev(np.zeros((1, 1), np.int32)), to_dev(slots),
                         validate_slots=False)
    wk, wv = np.zeros((nb, bs, H, D), np.float16), np.zeros((nb, bs, H, D), np.float16)
    live = slots < nb * bs
    O.write_cache(wk, k[live], slots[live])
    O.write_cache(wv, v[live], slots[live])
    same_bits(memopt_C.get_int4_pages(), O.to_int4_pages(wk, wv))
