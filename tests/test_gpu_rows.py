"""The row kernels at the sizes where their variants meet, each held to the
bits of another route to the same result: a long store's pages against the
same rows stored a page at a time, RoPE of many tokens against one token at a
time and against the table, the fold against the oracle's."""

import numpy as np
import pytest

from conftest import announce, fp16_exact
from oracle import ewma
from test_gpu_kv_pages import LAYERS, mi, normal, pages_for, put

pytestmark = pytest.mark.gpu

P = 32


@pytest.mark.parametrize("kv,hd,runs", [
    (8, 64, [65]),                 # few pages: job by job
    (8, 64, [P * 24]),             # the most pages as jobs
    (8, 64, [P * 24 + 1]),         # the shortest run, and a row over
    (2, 128, [7, P * 24 - 6, 33]), # a first page begun by an earlier store
    (2, 64, [31, 1, 96, P * 25]),
    (2, 64, [P * 256 + 5]),        # a full launch of pages
    (2, 64, [3, P * 257 + 40]),    # one page into a second launch
    (1, 64, [200]),                # not a register-quantiser shape
])
def test_a_long_store_is_its_pages_stored_one_at_a_time(kv, hd, runs):
    """Every page, the last of which a further store completes: its first
    rows have waited in an open page."""
    seq = sum(runs)
    pages = -(-seq // P)
    rng = np.random.default_rng(seq)
    k, v = normal(rng, pages * P, kv, hd), normal(rng, pages * P, kv, hd)
    tmap = [[(1, 0, 3, 2)[(p + l) % 4] for p in range(pages)] for l in range(LAYERS)]
    made = []
    for pieces in (list(runs), [min(P, seq - at) for at in range(0, seq, P)]):
        alloc, cache = pages_for(P, kv, hd, 0, tier_map=tmap, always_seal=True,
                                 capacity=pages * LAYERS + 8)
        announce("store", kv, hd, pieces[:4])
        cache.reserve(pages * P)
        at = 0
        for n in pieces + [pages * P - seq]:
            if n > 0:
                cache.store(1, put(k[at:at + n]), put(v[at:at + n]), at, n)
            at += n
        made.append([alloc.read(1, p) for p in range(pages)])
    for p, (a, b) in enumerate(zip(*made)):
        np.testing.assert_array_equal(a, b, err_msg=f"page {p}")


@pytest.mark.parametrize("seq,heads,hd", [
    (32, 32, 64), (33, 32, 64),    # the last token by token a pair, the first by workgroups
    (5, 3, 6), (700, 3, 34), (70, 2, 514), (40, 5, 1030),
    (600, 4, 64), (600, 5, 64), (600, 2, 128), (600, 3, 128),  # few heads: a thread a pair
])
def test_rope_of_many_tokens_is_each_tokens(seq, heads, hd):
    m = mi()
    d = m.device
    rng = np.random.default_rng(hd)
    x = fp16_exact(rng.standard_normal((seq, heads, hd)))
    positions = rng.integers(0, 3000, seq).astype(np.int32)
    dx, out = put(x), d.empty(x.size)
    announce("rope", seq, heads, hd)
    d.rope(dx, d.DeviceIndex(positions), out, seq, heads, hd, 1e6)
    got = out.raw().reshape(x.shape)
    table = d.RopeTable(hd, 1e6)
    table.cover(3000)
    for shift in (0, 1):  # 16-byte aligned rows, and rows two bytes off
        src = put(np.concatenate([np.zeros(shift), x.reshape(-1)]))
        dst = d.empty(x.size + shift)
        d.rope_from_table(d.view(src, shift, x.size), d.DeviceIndex(positions), table,
                          d.view(dst, shift, x.size), seq, heads, hd)
        np.testing.assert_array_equal(dst.raw()[shift:].reshape(x.shape).view(np.uint16),
                                      got.view(np.uint16))
    row = d.empty(heads * hd)
    for t in (0, seq // 2, seq - 1):
        d.rope(d.view(dx, t * heads * hd, heads * hd), d.DeviceIndex(positions[t:t + 1]), row, 1,
               heads, hd, 1e6)
        np.testing.assert_array_equal(row.raw().reshape(heads, hd).view(np.uint16),
                                      got[t].view(np.uint16))


@pytest.mark.parametrize("heads", [1, 7, 8, 9, 16, 23])
def test_the_fold_of_any_number_of_heads(heads):
    m = mi()
    d = m.device
    pages = 301
    rng = np.random.default_rng(heads)
    scores = d.ImportanceScores(2, pages + 3)
    steps = []
    for i in range(3):
        mass = rng.random((heads, pages)).astype(np.float32)
        announce("fold", heads, i)
        scores.fold(1, d.upload_f32(mass), heads, pages)
        steps.append((1, mass))
    np.testing.assert_array_equal(scores.download(), ewma.host_ewma(steps, 2, pages + 3))
