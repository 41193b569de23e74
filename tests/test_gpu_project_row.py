"""One row's projections through the matrix-vector kernel (linear.cpp): the
input lengths where its runs, splits and dispatch end, the three output
forms, and the calls it leaves to hipBLASLt, against float64 products.

Tolerance: both sides' fp16 operands are exact in fp32 products, so an output
parts from the float64 sum by the fp32 additions (at most one rounding of
2^-24 a term over the sum of magnitudes) and, for fp16 outputs, the one
rounding to 11 bits."""

import numpy as np
import pytest

from conftest import announce, fp16_exact
from test_gpu_kv_pages import mi, put

pytestmark = pytest.mark.gpu


def check(got, x, w, add, half):
    want = w.astype(np.float64) @ x.astype(np.float64) + add
    size = np.abs(w).astype(np.float64) @ np.abs(x).astype(np.float64) + np.abs(add)
    bound = x.size * 2.0**-24 * size + (2.0**-11 * np.abs(want) + 2.0**-24 if half else 0.0)
    assert (np.abs(got - want) <= bound).all(), np.max(np.abs(got - want) / bound)


@pytest.mark.parametrize("n_in,n_out", [
    (8, 1), (8, 5), (504, 7), (512, 4), (520, 1000), (1536, 256), (1536, 8960), (4096, 33),
    (64, 259), (64, 260), (504, 2020), (512, 4103), (512, 4104),  # many short rows: hipBLASLt's
    (1528, 12240), (1536, 12300),
    (4104, 9),       # the first length split over four waves
    (8960, 130), (16384, 6), (16392, 3), (32768, 5),
    (32776, 3), (12, 6), (1000, 3),   # hipBLASLt's: too long, not a multiple of 8 (1000 is)
])
def test_one_row_against_float64(n_in, n_out):
    m = mi()
    d = m.device
    rng = np.random.default_rng(n_in + n_out)
    x = fp16_exact(rng.standard_normal(n_in))
    w = fp16_exact(rng.standard_normal((n_out, n_in)) / np.sqrt(n_in))
    b = fp16_exact(rng.standard_normal(n_out))
    dx, dw, db = put(x), put(w), put(b)
    for bias in (None, db):
        announce("one row", n_in, n_out, "bias" if bias is not None else "")
        out = d.empty(n_out)
        d.linear(dx, dw, bias, out, 1, n_in, n_out)
        check(out.to_numpy(), x, w, b if bias is not None else np.zeros(n_out), True)
    start = rng.standard_normal(n_out).astype(np.float32)
    out = d.upload_f32(start)
    d.linear_accumulate(dx, dw, out, 1, n_in, n_out)
    check(out.to_numpy(), x, w, start.astype(np.float64), False)


def test_rows_off_their_alignment_and_several_rows_agree_with_one():
    """x and the weights 2 bytes off a 16-byte boundary (left to hipBLASLt),
    and the same row among others, give the row's products."""
    m = mi()
    d = m.device
    n_in, n_out = 256, 48
    rng = np.random.default_rng(4)
    x = fp16_exact(rng.standard_normal((3, n_in)))
    w = fp16_exact(rng.standard_normal((n_out, n_in)) / 16)
    dx, dw = put(x), put(w)
    shifted = put(np.concatenate([[0.0], x[1], [0.0], w.reshape(-1)]))
    for name, xs, ws, rows in (("several rows", dx, dw, 3),
                               ("x off", d.view(shifted, 1, n_in), dw, 1),
                               ("w off", d.view(dx, n_in, n_in),
                                d.view(shifted, n_in + 2, n_out * n_in), 1)):
        announce("alignment", name)
        out = d.empty(rows * n_out)
        d.linear(xs, ws, None, out, rows, n_in, n_out)
        got = out.to_numpy().reshape(rows, n_out)
        check(got[1 if rows == 3 else 0], x[1], w, np.zeros(n_out), True)


@pytest.mark.parametrize("hidden", [64, 1536])  # hipBLASLt's, and the matrix-vector kernel's
def test_logits_of_one_row(hidden):
    """The head's fp32 logits of one row among several, and its argmax."""
    m = mi()
    d = m.device
    vocab = 5003
    rng = np.random.default_rng(6)
    x = fp16_exact(rng.standard_normal((4, hidden)))
    w = fp16_exact(rng.standard_normal((vocab, hidden)) / np.sqrt(hidden))
    scratch = d.empty(d.scratch_elements(1, vocab))
    announce("logits of one row")
    got = d.logits(put(x), put(w), scratch, 2, 1, hidden, vocab)
    check(got[0], x[2], w, np.zeros(vocab), False)
    assert d.greedy(put(x), put(w), scratch, 2, 1, hidden, vocab)[0] == np.argmax(got[0])
