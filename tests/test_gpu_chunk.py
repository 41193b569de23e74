"""A long chunk's attention over laid-out pages (chunk.hip): the sizes where
its tiles, steps, splits and dispatch end, against the float64 oracle at the
attention gate (conftest.ATTN_MAX_REL, with the oracle's fp32 error bound)."""

import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from conftest import announce, assert_attention_close, fp16_exact
from oracle import attention as att
from test_gpu_kv_pages import mi, normal, pages_for, put, store_in_runs
from test_gpu_prefill import P, chunk_case

pytestmark = pytest.mark.gpu


def laid_out(cache) -> bool:
    return cache.chunk_scratch[0] == 1


@pytest.mark.parametrize("heads,kv,hd,seq,seq_q,bias,laid", [
    (32, 8, 64, P * 5 + 3, 143, False, False),   # over few keys: the most queries staged,
    (32, 8, 64, P * 5 + 3, 144, False, True),    # and the fewest laid out
    (12, 2, 128, P * 7 + 2, 191, True, False),
    (12, 2, 128, P * 7 + 2, 192, True, True),    # 21 queries a workgroup
    (32, 8, 64, 2049, 64, True, False),          # the same over many
    (32, 8, 64, 2049, 65, True, True),
    (12, 2, 128, 2049, 127, False, False),
    (12, 2, 128, 2049, 128, False, True),
    (12, 2, 128, 2048, 128, False, False),       # the most keys that are few
    (64, 8, 64, 127, 127, False, False),         # the most that are too few
    (64, 8, 64, 128, 128, False, True),          # a prompt of whole pages, nothing before it
    (32, 32, 128, P * 6, 127, False, False),     # a head a KV head: fewer rows than a workgroup's
    (32, 32, 128, P * 6, 128, True, True),
    (18, 18, 64, P * 9 + 1, 257, False, True),   # 256 queries a workgroup, and one
    (32, 8, 64, P * 7 + 31, 193, True, True),    # one query past three workgroups' 64
    (16, 1, 64, P * 10, 298, False, True),       # sixteen heads a KV head
    (14, 2, 64, P * 33 + 17, 330, True, True),   # rows that do not fill their tiles; splits
    (12, 2, 128, P * 40 + 30, 200, False, True),
    (12, 2, 128, P * 130 + 5, 128, True, True),  # many splits of few queries
])
def test_chunks_at_the_edges_of_tiles_steps_and_the_rule(heads, kv, hd, seq, seq_q, bias, laid):
    caches = []
    chunk_case(heads, kv, hd, seq, seq_q, 11, bias, True, caches=caches)
    assert laid_out(caches[0]) == laid


@pytest.mark.parametrize("hd,kv,heads", [(64, 8, 32), (128, 2, 12)])
@pytest.mark.parametrize("bias", [False, True])
def test_unread_pages_before_and_inside_a_long_chunk(hd, kv, heads, bias):
    """Masked pages, among them the first, two of one step, and sealed pages
    of the chunk's own positions."""
    caches = []
    chunk_case(heads, kv, hd, P * 14 + 9, 6 * P, 3, bias, False, (0, 4, 5, 7, 11, 12), caches)
    assert laid_out(caches[0])


@pytest.mark.parametrize("heads,kv,hd,seq_q", [(32, 8, 64, 150), (12, 2, 128, 200)])
def test_one_score_far_above_the_rest_moves_the_reference(heads, kv, hd, seq_q):
    """Scores that rise by hundreds of powers of two from one page to the
    next, and fall again: each row's softmax reference moves up step by step
    and its earlier sums vanish."""
    rng = np.random.default_rng(2)
    seq = P * 12 + 5
    k, v = normal(rng, seq, kv, hd), normal(rng, seq, kv, hd)
    q = normal(rng, seq_q, heads, hd)
    for page, size in ((1, 4.0), (3, 12.0), (4, 40.0), (8, 6.0)):
        k[page * P + 7] = size * np.sign(q[0, 0])
    fp16_case("chunk outlier scores", q, k, v)


def fp16_case(what, q, k, v, bias=None, theta=1e6):
    """The last queries' attention over a cache of FP16 pages, laid out, held
    to the oracle."""
    d = mi().device
    (seq, kv, hd), (seq_q, heads, _) = k.shape, q.shape
    alloc, cache = pages_for(P, kv, hd, 0)
    store_in_runs(cache, 0, k, v, [seq])
    rope = None
    if bias is not None:
        rope = d.RopeTable(hd, theta)
        rope.cover(seq)
    out = d.empty(q.size)
    announce(what, heads, kv, hd, seq, seq_q)
    cache.attention(0, put(q), put(bias) if bias is not None else None, rope, out, seq_q, seq,
                    heads, kv, hd, None, None, None, None)
    assert laid_out(cache)
    want, w = att.attention64(q, k, v, bias, theta)
    assert_attention_close(out.to_numpy().reshape(q.shape), want, what,
                           att.attention_bound(q, k, v, w, bias, theta))


@pytest.mark.parametrize("heads,kv,hd,seq_q", [(32, 8, 64, 170), (12, 2, 128, 200)])
def test_an_fp16_page_table_with_the_key_bias(heads, kv, hd, seq_q):
    rng = np.random.default_rng(4)
    seq = P * 11 + 20
    fp16_case("FP16 pages with the key bias", normal(rng, seq_q, heads, hd),
              normal(rng, seq, kv, hd), normal(rng, seq, kv, hd),
              fp16_exact(3 * rng.standard_normal((kv, hd))))


@pytest.mark.parametrize("heads,kv,hd,seq_q", [(32, 8, 64, 170), (12, 2, 128, 200)])
@pytest.mark.parametrize("page", [0, 3])  # the one that gives the first reference, and another
def test_infinite_keys_and_values_before_a_chunk(heads, kv, hd, seq_q, page):
    """One infinite element of a key: the rows whose score it makes -inf give
    it no weight, the others have no result. One infinite element of a value:
    its channel has none, every other is as it was."""
    rng = np.random.default_rng(page + 6)
    seq, at = P * 12 + 5, page * P + 9
    k, v = normal(rng, seq, kv, hd), normal(rng, seq, kv, hd)
    q = normal(rng, seq_q, heads, hd)
    q[:, :, 3] = np.where(q[:, :, 3] < 0, -1.0, 1.0)
    d = mi().device

    def attend(keys, values):
        alloc, cache = pages_for(P, kv, hd, 0)
        store_in_runs(cache, 0, keys, values, [seq])
        out = d.empty(q.size)
        announce("infinite", heads, kv, hd, page)
        cache.attention(0, put(q), None, None, out, seq_q, seq, heads, kv, hd, None, None, None,
                        None)
        assert laid_out(cache)
        return out.to_numpy().reshape(q.shape)

    group = heads // kv
    bad = k.copy()
    bad[at, 1, 3] = np.inf
    got = attend(bad, v)
    unread = np.arange(seq) == at
    want, w = att.attention64(q, k, v, unread=unread)
    full, wf = att.attention64(q, k, v)
    bound = att.attention_bound(q, k, v, w, unread=unread)
    bound_f = att.attention_bound(q, k, v, wf)
    reads = np.zeros(heads, bool)
    reads[group:2 * group] = True
    assert_attention_close(got[:, ~reads], full[:, ~reads], "other heads", bound_f[:, ~reads])
    none = reads[None, :] & (q[:, :, 3] > 0)
    assert not np.isfinite(got[none]).any()
    drops = reads[None, :] & (q[:, :, 3] < 0)
    assert_attention_close(got[drops], want[drops], "no weight", bound[drops])
    bad = v.copy()
    bad[at, 1, 5] = -np.inf
    got = attend(k, bad)
    hit = np.zeros((heads, hd), bool)
    hit[group:2 * group, 5] = True
    assert not np.isfinite(got[:, hit]).any()
    assert_attention_close(got[:, ~hit], full[:, ~hit], "other channels", bound_f[:, ~hit])


@pytest.mark.parametrize("heads,kv,hd,seq_q,high", [(32, 8, 64, 134, 2.162109375),
                                                       (12, 2, 128, 160, 1.509765625)])
def test_small_probabilities_keep_their_bits(heads, kv, hd, seq_q, high):
    """One key far above 8,191 others whose values are all the output: each of
    theirs is some 2^-25 of its weight, of which fp16 high and low parts of
    p x 2^14 hold 2^-14 at least (their last bit is 2^-38 of the weight; of
    p x 2^5 it would be 2^-29, a thirtieth of such a probability). Besides it
    the outputs part from float64 by the fp16 store's rounding and fp32
    exponents and sums (2^-16)."""
    seq = P * 256
    m = mi()
    d = m.device
    k, v = np.zeros((seq, kv, hd), np.float32), np.full((seq, kv, hd), 4096.0, np.float32)
    k[0], v[0] = high, 0.0
    q = np.ones((seq_q, heads, hd), np.float32)
    alloc, cache = pages_for(P, kv, hd, 0)
    store_in_runs(cache, 0, k, v, [seq])
    out = d.empty(q.size)
    announce("chunk small probabilities", heads, kv, hd)
    cache.attention(0, put(q), None, None, out, seq_q, seq, heads, kv, hd, None, None, None, None)
    assert laid_out(cache)
    keys = np.arange(seq - seq_q, seq)  # keys besides the first that a query reads
    weight = keys * np.exp(-high * np.sqrt(float(hd)))
    want = 4096.0 * weight / (1.0 + weight)
    got = out.to_numpy().reshape(seq_q, -1)
    error = np.abs(got / want[:, None] - 1.0).max()
    assert error < 2.0**-11 + 2.0**-14 + 2.0**-16, error


def chunk_call(layers=1, seq=P * 9 + 4, seq_q=144):
    """A cache of `seq` positions and call(layer, out): its last seq_q
    queries' attention; and each layer's attention and error bound."""
    m = mi()
    d = m.device
    heads, kv, hd = 32, 8, 64
    rng = np.random.default_rng(9)
    q = normal(rng, seq_q, heads, hd)
    alloc, cache = pages_for(P, kv, hd, 0)
    exact = []
    for layer in range(layers):
        k, v = normal(rng, seq, kv, hd), normal(rng, seq, kv, hd)
        store_in_runs(cache, layer, k, v, [seq])
        want, w = att.attention64(q, k, v)
        exact.append((want, att.attention_bound(q, k, v, w)))
    dq = put(q)

    def call(layer, out, queries=seq_q):
        cache.attention(layer, dq, None, None, out, queries, seq, heads, kv, hd, None, None, None,
                        None)

    def check(out, layer, what):
        want, bound = exact[layer]
        assert_attention_close(out.to_numpy().reshape(q.shape), want, what, bound)

    for layer in range(layers):
        call(layer, d.empty(q.size), 2)  # the page table is sent
    m.synchronize()
    assert cache.chunk_scratch == (0, 0)
    return (alloc, cache), call, lambda: d.empty(q.size), check


def test_a_captured_chunk_takes_the_staging_path():
    """A captured launch gets no scratch: the graph replayed between the
    program's own calls, which do."""
    m = mi()
    d = m.device
    (_, cache), call, empty, check = chunk_call()
    out = empty()
    stream = m.Stream()
    graph = m.Graph(stream)
    with graph.capture():
        call(0, out)
    assert cache.chunk_scratch == (0, 0)
    for i in range(3):
        announce("chunk graph replay", i)
        d.random_half(out, 70 + i, 1.0)
        m.synchronize()
        graph.launch()
        stream.synchronize()
        check(out, 0, f"replay {i}")
        d.random_half(out, 90 + i, 1.0)
        call(0, out)
        check(out, 0, f"eager {i}")
        assert cache.chunk_scratch[0] == i + 1


def test_a_chunk_while_its_thread_captures_another_stream():
    """The scratch's allocation and its return neither fail for a capture on
    another stream nor spoil it."""
    m = mi()
    d = m.device
    (_, cache), call, empty, check = chunk_call()
    outs = [empty(), empty()]
    side, stream = m.Stream(), m.Stream()
    x, y = put(np.ones(64, np.float32)), put(np.ones(64, np.float32))
    graph = m.Graph(stream)
    with graph.capture():
        d.add(x, y, x, 64)
        m.set_stream(side)
        for out in outs:
            announce("chunk beside a capture")
            call(0, out)
            assert m.release_chunk_scratch() > 0
        m.set_stream(stream)
        d.add(x, y, x, 64)
    side.synchronize()
    for out in outs:
        check(out, 0, "beside a capture")
    assert cache.chunk_scratch == (2, 0)
    for i in range(3):
        graph.launch()
        stream.synchronize()
        np.testing.assert_array_equal(x.to_numpy(), np.full(64, 3.0 + 2 * i))


def test_every_stream_lays_its_pages_out_in_the_one_scratch():
    """Chunks of two layers on streams that come and go, more than any fixed
    number, none waited for in between: each waits for the chunk before it."""
    m = mi()
    d = m.device
    (_, cache), call, empty, check = chunk_call(layers=2, seq=P * 40 + 4)
    outs = [empty() for _ in range(12)]
    keep = [m.Stream() for _ in range(3)]
    for i, out in enumerate(outs):
        announce("chunk stream", i)
        stream = keep[i % 3] if i % 2 else m.Stream()
        m.set_stream(stream)
        try:
            call(i % 2, out)
        finally:
            m.set_stream(None)
    m.synchronize()
    for i, out in enumerate(outs):
        check(out, i % 2, f"call {i}")
    assert cache.chunk_scratch[0] == len(outs)


def test_the_scratch_is_given_back():
    m = mi()
    (_, cache), call, empty, check = chunk_call()
    m.release_chunk_scratch()
    out = empty()
    call(0, out)
    held = cache.chunk_scratch[1]
    assert held > 0
    assert m.release_chunk_scratch() == held
    assert cache.chunk_scratch == (1, 0)
    check(out, 0, "before")
    call(0, out)
    check(out, 0, "after")
    assert cache.chunk_scratch == (2, held)


def test_two_threads_chunks_on_one_stream_keep_their_own_layout():
    """Chunks of two layers from two threads, both on the null stream: the
    scratch is the stream's, so each chunk's launches follow the other's
    whole. Every output has the bits of the call by itself."""
    m = mi()
    d = m.device
    heads, kv, hd, seq, seq_q, calls = 32, 8, 64, P * 40 + 4, 160, 24
    rng = np.random.default_rng(5)
    alloc, cache = pages_for(P, kv, hd, 0)
    for layer in (0, 1):
        store_in_runs(cache, layer, normal(rng, seq, kv, hd), normal(rng, seq, kv, hd), [seq])
    dq = put(normal(rng, seq_q, heads, hd))
    n = seq_q * heads * hd

    def attend(layer, out):
        cache.attention(layer, dq, None, None, out, seq_q, seq, heads, kv, hd, None, None, None,
                        None)

    want = []
    for layer in (0, 1):
        out = d.empty(n)
        attend(layer, out)
        want.append(out.to_numpy())
    outs = [[d.empty(n) for _ in range(calls)] for _ in (0, 1)]
    start = threading.Barrier(2)

    def work(layer):
        start.wait()
        for out in outs[layer]:
            attend(layer, out)

    announce("chunks from two threads")
    with ThreadPoolExecutor(2) as pool:
        list(pool.map(work, (0, 1)))
    m.synchronize()
    for layer in (0, 1):
        for i, out in enumerate(outs[layer]):
            assert np.array_equal(out.to_numpy(), want[layer]), (layer, i)
    assert cache.chunk_scratch[0] == 2 + 2 * calls
