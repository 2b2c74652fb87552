"""Logits of layer-list prompts on their way to the caller (csrc/kh_model_step.hip, logits_pin): any number of rows, growing and falling,
through the pinned buffer and beside it, and what a call costs that wants more rows than any before it."""
import time

import numpy as np
import pytest

import layers_util as U

pytestmark = pytest.mark.gpu


def _model(vocab, **kw):
    mod = U.Model(U.config([U.mamba()], width=48, vocab=vocab))
    return mod, mod.load("float32", max_seq_len=128, **kw)


@pytest.mark.parametrize("vocab", [101, 32000])
def test_rows_of_any_number(gpu, vocab):
    """33 rows of 32000 are more than the 4 MB that go through pinned memory."""
    mod, m = _model(vocab)
    toks = mod.tokens(40)
    ref = mod.logits(toks)
    for n in (1, 2, 3, 5, 9, 33, 4, 32, 40, 1):
        s = m.open_seq()
        U.check(m.forward([(s, toks, list(range(40 - n, 40)))]), ref[40 - n:], "float32", n)
        m.close_seq(s)
    m.close()


def test_one_row_more_costs_no_allocation(gpu):
    """A buffer grown row by row made every such call several times as long as the next one like it; grown to powers of two it is
    four calls of fourteen."""
    mod, m = _model(32000)
    toks = mod.tokens(40)

    def once(n):
        s = m.open_seq()
        t = time.perf_counter()
        m.forward([(s, toks, list(range(40 - n, 40)))])
        t = time.perf_counter() - t
        m.close_seq(s)
        return t

    s = m.open_seq()
    m.forward([(s, toks, [])])
    m.close_seq(s)
    ratio = []
    for n in range(2, 16):
        first = once(n)
        ratio.append(first / np.median([once(n) for _ in range(7)]))
    m.close()
    print(np.round(ratio, 2))
    assert np.median(ratio) < 1.7
