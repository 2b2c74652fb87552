"""The last layer of a pass for its wanted tokens alone (csrc/kh_hybrid_step.hip, hy_tail) against the plain reference: every kind
of last layer, loops that end there, wanted rows inside a sequence, sequences of unequal length, and what follows."""
import numpy as np
import pytest

import layers_util as U
from kuiperllama_amd import _ffi

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])

CASES = {
    "mamba": U.config([U.with_ff(U.latent()), U.with_ff(U.mamba(inner=130, state=20, dt_rank=7, conv=3))]),
    "mamba-shared-only": U.config([U.mamba(), U.with_ff(U.mamba(), experts=3, identity=0, top=3, shared=33)]),
    "mamba-no-ff": U.config([U.mamba(), U.mamba(33, 1, 1, 1)]),
    "latent": U.config([U.with_ff(U.mamba()), U.with_ff(U.latent(2, 36, 8, 16, 70, 50, 0.4), identity=0, shared=0, top=2)]),
    "window": U.gusorax([dict(U.chunked(), mlp=U.clamped()), dict(U.windowed(), mlp=U.dense())]),
    "chunk": U.gusorax([dict(U.windowed(), mlp=U.dense()), dict(U.chunked(), mlp=U.clamped())]),
    "loop-to-the-end": U.config([U.with_ff(U.mamba()), U.with_ff(U.latent()), U.mamba(40, 17, 3, 3)], loop=(1, 3, 2)),
    "loop-of-the-last": U.config([U.with_ff(U.latent()), U.with_ff(U.mamba())], loop=(1, 2, 3)),
    "matrix-loop-to-the-end": U.gusorax([dict(U.windowed(), mlp=U.dense()), dict(U.chunked(), mlp=U.clamped())], loop=(1, 2, 2)),
    "one-layer": U.config([U.with_ff(U.latent())]),
}


@pytest.fixture(params=sorted(CASES))
def mod(request):
    return U.Model(CASES[request.param], seed=5)


@BOTH
def test_last_token_and_what_follows(gpu, mod, dtype):
    for n in (4, 37, 133):
        toks = mod.tokens(n + 3)
        ref = mod.logits(toks)
        m = mod.load(dtype)
        s = m.open_seq()
        got = [m.forward([(s, toks[:n], [n - 1])])]
        got += [m.forward([(s, [t], [0])]) for t in toks[n:]]
        m.close()
        U.check(np.concatenate(got), ref[n - 1:], dtype, n)


@BOTH
def test_rows_inside_and_unequal_sequences(gpu, mod, dtype):
    lens, wants = (70, 9, 141), ([69], [], [3, 140])
    m = mod.load(dtype)
    toks = [mod.tokens(n + 1, seed=n) for n in lens]
    seqs = [m.open_seq() for _ in lens]
    got = m.forward([(s, t[:n], w) for s, t, n, w in zip(seqs, toks, lens, wants)])
    more = m.forward([(s, [t[n]], [0]) for s, t, n in zip(seqs, toks, lens)])
    m.close()
    refs = [mod.logits(t) for t in toks]
    U.check(got, np.concatenate([r[w] for r, w in zip(refs, wants) if w]), dtype, "pass")
    U.check(more, np.stack([r[n] for r, n in zip(refs, lens)]), dtype, "step")


def test_same_as_the_whole_layer_and_over_passes(gpu):
    """fp32: hook off, on, and a prompt cut into passes, whose last one alone has a wanted row; the logits' spread is one."""
    for name in ("mamba", "latent", "chunk"):
        mod = U.Model(CASES[name], seed=6)
        toks = mod.tokens(150)
        out = {}
        for hooks in ((), (("KH_HY_TAIL", "0"),), (("KH_HY_TMAX", "64"),)):
            for k, v in hooks:
                _ffi.debug_set(k, v)
            try:
                m = mod.load("float32")
                s = m.open_seq()
                out[hooks] = m.forward([(s, toks, [149])])
                m.close()
            finally:
                for k, _ in hooks:
                    _ffi.debug_set(k, None)
        U.check(out[()], mod.logits(toks)[149:], "float32", name)
        for o in out.values():
            assert np.abs(o - out[()]).max() <= 2e-4 * np.abs(out[()]).max(), name
