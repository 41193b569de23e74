"""One layer's decode where its split changes: a quarter of a workgroup's
waves a split, half of them up to a workgroup a CU, all of them past it. Outputs
and masses against the float64 oracle on both sides; a launch sized for a long
context with its seq_k on the device, and the statistics kept for a later fold,
to the bits of the plain launch at every seq_k; a run of steps across a change
to the bits of the steps one by one, whose kernels are chosen by their own
positions."""

import numpy as np
import pytest

from conftest import announce, assert_attention_close, fp16_exact
from oracle import attention as att
from oracle import ewma
from test_gpu_decode_step import (context_rows, make_cache, make_weights, prefill, small_shape,
                                  tier_map_for, upload_weights)
from test_gpu_kv_pages import LAYERS, mi, normal, page_sizes, put, sealed_pages

pytestmark = pytest.mark.gpu

P = 32
THETA = 1e6


def cache_of(seq, kv, hd, most):
    m = mi()
    pages = most // P + 1
    tmap = [[(1, 0, 3, 2)[(p + l) % 4] for p in range(pages)] for l in range(LAYERS)]
    cap = [pages * LAYERS + 16] * 4
    alloc = m.PagedKVCache(page_sizes(P, kv, hd), cap)
    cache = m.device.KVPages(alloc, LAYERS, P, kv, hd, 0, m.device.Halves.Both, tmap, True)
    cache.reserve(most)
    return alloc, cache


@pytest.mark.parametrize("heads,kv,hd,bias", [(12, 2, 128, False), (12, 2, 128, True),
                                              (14, 2, 64, True), (32, 8, 64, False),
                                              (5, 1, 128, False)])
def test_decode_on_both_sides_of_the_split(heads, kv, hd, bias):
    m = mi()
    d = m.device
    # The pages past which splits of two would make more than five workgroups
    # for eight CUs, and of four more than one a CU (256 CUs).
    two = 160 // kv * 2 * P
    edge = 256 // kv * 4 * P
    most = edge + 3 * P
    rng = np.random.default_rng(heads + hd + bias)
    k, v = normal(rng, most, kv, hd), normal(rng, most, kv, hd)
    b = fp16_exact(3 * rng.standard_normal((kv, hd))) if bias else None
    db = put(b) if bias else None
    rope = d.RopeTable(hd, THETA) if bias else None
    if bias:
        rope.cover(most)
    part = d.empty_f32(d.attention_partials(hd))
    q = [put(normal(rng, heads, hd)) for _ in range(LAYERS)]
    for seq in (1, P + 1, 5 * P, two, two + 1, edge, edge + 1, edge + 2 * P + 7):
        alloc, cache = cache_of(seq, kv, hd, most)
        for l in range(LAYERS):
            if seq > 1:
                cache.store(l, put(k[:seq - 1]), put(v[:seq - 1]), 0, seq - 1)
            cache.store(l, put(k[seq - 1:seq]), put(v[seq - 1:seq]), seq - 1, 1)
        kr, vr = put(k[seq - 1:seq]), put(v[seq - 1:seq])
        pages = -(-seq // P)
        masses, outs = [], []
        for l in range(LAYERS):
            announce("decode", heads, kv, hd, "bias" if bias else "", seq, l)
            out, mass = d.empty(heads * hd), d.empty_f32(heads * pages)
            cache.attention(l, q[l], db, rope, out, 1, seq, heads, kv, hd, kr, vr, mass, part)
            outs.append(out.raw())
            masses.append(mass.to_numpy())
            live = d.empty(heads * hd)
            cache.attention_at(l, q[l], db, rope, live, d.DeviceIndex([seq]), most, heads, kv, hd,
                               kr, vr)
            np.testing.assert_array_equal(live.raw().view(np.uint16), outs[l].view(np.uint16))
        kept = d.empty(heads * hd)
        for l in range(LAYERS):
            cache.attention_kept(l, q[l], db, rope, kept, seq, heads, kv, hd, kr, vr)
            np.testing.assert_array_equal(kept.raw().view(np.uint16), outs[l].view(np.uint16))
        scores = d.ImportanceScores(LAYERS, pages)
        mass = d.empty_f32(LAYERS * heads * pages)
        cache.fold_kept(scores=scores, mass=mass, seq_k=seq, heads=heads)
        got = mass.to_numpy().reshape(LAYERS, heads, pages)
        np.testing.assert_array_equal(got, np.stack(masses).reshape(got.shape))
        np.testing.assert_array_equal(
            scores.download(), ewma.host_ewma([(l, got[l]) for l in range(LAYERS)], LAYERS, pages))
        sealed, tiers = sealed_pages(alloc, 0, (seq - 1) // P)
        want, bound = att.causal_chunk(q[0].raw().reshape(1, heads, hd).astype(np.float32), sealed,
                                       tiers, k[:seq], v[:seq], kv, hd, P, b, THETA,
                                       with_bound=True)
        assert_attention_close(outs[0].astype(np.float64).reshape(1, heads, hd), want,
                               f"seq {seq}", bound)
        np.testing.assert_allclose(got[0].sum(1), 1.0, rtol=1e-3)


@pytest.mark.parametrize("start", [
    60,    # from two pages, one split either way, to three
    1020,  # from 32 pages, splits of four, to 33, splits of eight
])
@pytest.mark.parametrize("bias", [False, True])
def test_a_run_across_a_change_of_split_is_its_steps(start, bias):
    """32 KV heads: splits of two up to 10 pages, of four up to 32 (256 CUs).
    (Steps launched from the host: the launches a graph would hold.)"""
    m = mi()
    d = m.device
    s = small_shape(heads=32, kv_heads=32, head_dim=64)
    rng = np.random.default_rng(start)
    dev = upload_weights(make_weights(rng, s, bias))
    rows = context_rows(rng, s, start)
    n, made = 9, []
    for runs in ([n], [1] * n):
        alloc, cache = make_cache(s, tier_map_for(s, 64))
        prefill(cache, s, rows)
        scores = d.ImportanceScores(s["layers"], 40)
        step = d.DecodeStep(cache, s, dev["embed"], dev["final_norm"], dev["head"], dev["layers"],
                            scores, 1)
        token, at, tokens = 3, start, []
        for k in runs:
            announce("steps across a split", start, bias, at, k)
            out, _ = step.run(token, at, k, graphed=False)
            tokens += [int(t) for t in out]
            token, at = tokens[-1], at + k
        made.append((tokens, step.logits(), scores.download(), alloc, cache, step))
    assert made[0][0] == made[1][0]
    np.testing.assert_array_equal(made[0][1], made[1][1])
    np.testing.assert_array_equal(made[0][2], made[1][2])
