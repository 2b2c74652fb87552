"""Several wanted tokens of one sequence in the last layer's step behind a pass (csrc/kh_hybrid_step.hip, hy_tail), where that layer
attends over heads: one token sees another's cache row, which that one's step writes.  Two and four places of one sequence, two
sequences of two, in a window, a chunk and beyond them: against the plain reference and the whole layer, the same bits every time."""
import numpy as np
import pytest

import layers_util as U
from kuiperllama_amd import _ffi

pytestmark = pytest.mark.gpu
KW = dict(heads=8, kv_heads=2, dim=128, vdim=64, scale=128 ** -0.5)
LAST = {"window": dict(U.windowed(window=40, rows=16, far=90.0, **KW), mlp=U.clamped()),
        "chunk": dict(U.chunked(chunk=400, **KW), mlp=U.clamped(16, 6, 64)),
        "dense": dict(U.chunked(chunk=64, heads=3, kv_heads=3, dim=50, vdim=70, scale=0.15), mlp=U.dense())}
WANTS = [[(64, [10, 63])], [(141, [3, 140])], [(141, [96, 97, 98, 99])], [(100, [0, 31, 64, 99])], [(70, [20, 69]), (90, [50, 51])]]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("last", sorted(LAST))
def test_tokens_of_one_sequence(gpu, dtype, last):
    mod = U.Model(U.gusorax([dict(U.windowed(), mlp=U.dense()), LAST[last]]), seed=3)
    for want in WANTS:
        toks = [mod.tokens(n + 1, seed=10 * n + i) for i, (n, _) in enumerate(want)]
        refs = [mod.logits(t) for t in toks]
        out = {}
        for hook in (None, "0"):
            _ffi.debug_set("KH_HY_TAIL", hook)
            try:
                m = mod.load(dtype)
                for _ in range(6):
                    seqs = [m.open_seq() for _ in want]
                    got = m.forward([(s, t[:n], w) for s, t, (n, w) in zip(seqs, toks, want)])
                    more = m.forward([(s, t[n:], [0]) for s, t, (n, _) in zip(seqs, toks, want)])
                    for s in seqs:
                        m.close_seq(s)
                    out.setdefault(hook, []).append((got, more))
                m.close()
            finally:
                _ffi.debug_set("KH_HY_TAIL", None)
            for got, more in out[hook]:
                np.testing.assert_array_equal(got, out[hook][0][0])
                np.testing.assert_array_equal(more, out[hook][0][1])
            U.check(out[hook][0][0], np.concatenate([r[w] for r, (_, w) in zip(refs, want)]), dtype, f"{want} {hook}")
            U.check(out[hook][0][1], np.stack([r[n] for r, (n, _) in zip(refs, want)]), dtype, f"{want} {hook} step")
