"""Mixers of a pass beside its feed-forwards on a second stream (csrc/kh_hybrid_pass.hip, Runner::fork): the same kernels on the same
inputs, so the same bits as on one stream - prompts, pieces behind others, several passes a call, two sequences, a loop."""
import numpy as np
import pytest

import layers_util as U
from kuiperllama_amd import _ffi

pytestmark = pytest.mark.gpu


def _gufanex():
    moe = dict(experts=32, identity=4, top=6, ff=512)
    return U.config([U.with_ff(U.mamba(1024, 8, 16, 4), **moe), U.with_ff(U.latent(4, 64, 32, 64, 128, 256, 0.1), **moe)], width=1024,
                    vocab=300, loop=(0, 1, 2))


def _gusorax():
    kw = dict(heads=8, kv_heads=2, dim=128, vdim=128, scale=128 ** -0.5)
    moe = U.clamped(experts=32, top=7, ff=512)
    return U.gusorax([dict(U.windowed(window=100, rows=16, far=90.0, **kw), mlp=moe), dict(U.chunked(chunk=120, **kw), mlp=moe)],
                     width=1024, vocab=300, positions=600)


def _dense():
    kw = dict(heads=8, kv_heads=2, dim=64, vdim=64, scale=0.125)
    return U.gusorax([dict(U.windowed(window=100, rows=16, far=90.0, **kw), mlp=U.dense(1024)), dict(U.chunked(chunk=120, **kw), mlp=U.dense(40))],
                     width=512, vocab=300, positions=600)


@pytest.mark.parametrize("arch,dtype", [(_gufanex, "bfloat16"), (_gusorax, "bfloat16"), (_gusorax, "float32"), (_dense, "float32")])
def test_same_bits_as_on_one_stream(gpu, arch, dtype, monkeypatch):
    """Every layer on one stream, every layer on two, and as the rule has it."""
    mod = U.Model(arch())
    toks = mod.tokens(300)
    monkeypatch.setenv("KH_HY_TMAX", "128")
    m = mod.load(dtype, max_seqs=2)

    def run(fork):
        _ffi.debug_set("KH_HY_FORK", fork)
        assert _ffi.debug_get("KH_HY_FORK") == fork
        out = [U.run_alone(m, toks, (17, 19, 150))]  # 131 and 150 tokens: two passes each
        a, b = m.open_seq(), m.open_seq()
        out.append(m.forward([(a, toks[:90], [0, 50, 89]), (b, toks[40:100], [59])]))
        out.append(m.forward([(a, toks[90:94], [3]), (b, toks[100:260], [0, 159])]))
        m.close_seq(a)
        m.close_seq(b)
        return out

    try:
        want = run("0")
        U.check(want[0], mod.logits(toks), dtype, "one stream")
        for fork in ("1", None, "1", None, "1"):
            for x, y in zip(run(fork), want):
                np.testing.assert_array_equal(x, y)
    finally:
        _ffi.debug_set("KH_HY_FORK", None)
        m.close()
