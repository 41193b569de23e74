"""A long chunk's attention over laid-out pages (chunk.hip): the sizes where
its tiles, steps, splits and dispatch end, against the float64 oracle at the
attention gate (conftest.ATTN_MAX_REL, with the oracle's fp32 error bound)."""

import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from conftest import announce, assert_attention_close
from oracle import attention as att
from test_gpu_kv_pages import mi, normal, pages_for, put, store_in_runs
from test_gpu_prefill import P, chunk_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,hd,seq,seq_q,bias", [
    (32, 8, 64, P * 5 + 3, 127, False),     # the largest chunk that stages page by page
    (32, 8, 64, P * 5 + 3, 128, False),     # the smallest over laid-out pages
    (32, 8, 64, 128, 128, False),            # a prompt of whole pages, nothing before it
    (32, 8, 64, P * 7 + 31, 129, True),     # one query past two workgroups' 64
    (4, 4, 64, P * 9 + 1, 257, False),     # a head a KV head: 256 queries a workgroup, and one
    (16, 1, 64, P * 6, 154, False),         # sixteen heads a KV head
    (14, 2, 64, P * 33 + 17, 137, True),    # rows that do not fill their tiles; steps in splits
    (12, 2, 128, P * 3 + 2, 64, True),     # head_dim 128: 21 queries a workgroup
    (12, 2, 128, P * 40 + 30, 150, False),
    (12, 2, 128, P * 130 + 5, 64, True),   # many splits of few queries
    (8, 8, 128, P * 4 + 9, 129, False),
])
def test_chunks_at_the_edges_of_tiles_and_steps(heads, kv, hd, seq, seq_q, bias):
    chunk_case(heads, kv, hd, seq, seq_q, 11, bias, True)


@pytest.mark.parametrize("hd,kv,heads", [(64, 8, 32), (128, 2, 12)])
def test_unread_pages_before_and_inside_a_long_chunk(hd, kv, heads):
    """Masked pages, among them the first, two of one step, and sealed pages
    of the chunk's own positions."""
    seq, seq_q = P * 14 + 9, 4 * P
    chunk_case(heads, kv, hd, seq, seq_q, 3, False, False, (0, 4, 5, 7, 11, 12))


@pytest.mark.parametrize("heads,kv,hd", [(32, 8, 64), (12, 2, 128)])
def test_one_score_far_above_the_rest_moves_the_reference(heads, kv, hd):
    """Scores that rise by hundreds of powers of two from one page to the
    next, and fall again: each row's softmax reference moves up step by step
    and its earlier sums vanish."""
    rng = np.random.default_rng(2)
    seq, seq_q = P * 12 + 5, 134
    k, v = normal(rng, seq, kv, hd), normal(rng, seq, kv, hd)
    q = normal(rng, seq_q, heads, hd)
    for page, size in ((1, 4.0), (3, 12.0), (4, 40.0), (8, 6.0)):
        k[page * P + 7] = size * np.sign(q[0, 0])
    m = mi()
    d = m.device
    alloc, cache = pages_for(P, kv, hd, 0)
    store_in_runs(cache, 0, k, v, [seq])
    out = d.empty(q.size)
    announce("chunk outlier scores", heads, kv, hd)
    cache.attention(0, put(q), None, None, out, seq_q, seq, heads, kv, hd, None, None, None, None)
    want, w = att.attention64(q, k, v)
    assert_attention_close(out.to_numpy().reshape(q.shape), want, "outliers",
                           att.attention_bound(q, k, v, w))


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
    heads, kv, hd, seq, seq_q, calls = 32, 8, 64, P * 40 + 4, 128, 24
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
