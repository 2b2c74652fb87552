"""Attention over heads beside the experts of a decode step (csrc/kh_ldheads.h) against the plain reference and against the
launches of its own (hook KH_HY_BESIDE=0): edges of its splits, tiles and steps of 16 keys, groups of more and fewer heads than
four, padded and full sizes, a ring that wraps, one to four sequences."""
import numpy as np
import pytest

import layers_util as U
from kuiperllama_amd import _ffi

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])


@pytest.fixture
def own_launches():
    def set_(on):
        _ffi.debug_set("KH_HY_BESIDE", "0" if on else None)
    yield set_
    _ffi.debug_set("KH_HY_BESIDE", None)


def steps(m, toks, at, n):
    """Logits of n steps of one sequence for each start in `at`, up to four at once."""
    seqs = [m.open_seq() for _ in at]
    for s, k in zip(seqs, at):
        if k:
            m.forward([(s, toks[:k], [])])
    out = [m.forward([(s, [toks[k + i]], [0]) for s, k in zip(seqs, at)]) for i in range(n)]
    for s in seqs:
        m.close_seq(s)
    return np.stack(out, 1)


@BOTH
@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(8, 2, 128, 128), (5, 1, 128, 64), (3, 3, 64, 128), (16, 1, 50, 120),
                                                    (9, 1, 127, 65), (2, 1, 1, 3)])
def test_against_launches_of_its_own(gpu, dtype, heads, kv_heads, dim, vdim, own_launches):
    """Splits of 32 keys (bf16: 64), two of them, 16 of them, longer ones, and whatever the window leaves of a ring that wraps."""
    kw = dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, scale=dim ** -0.5)
    mod = U.Model(U.gusorax([dict(U.windowed(window=300, rows=16, far=90.0, **kw), mlp=U.clamped()), U.chunked(chunk=1200, **kw),
                             U.windowed(window=2000, rows=32, far=1500.0, **kw)], positions=2000))
    toks = mod.tokens(1290)
    want = mod.logits(toks)
    starts = [[0, 15, 31, 63], [126, 299, 510, 1022], [1198], [1278, 1150]]
    for on in (False, True):
        own_launches(on)
        m = mod.load(dtype, max_seq_len=1800, max_seqs=4)
        for at in starts:
            got = steps(m, toks, at, 4)
            for k, g in zip(at, got):
                U.check(g, want[k: k + 4], dtype, f"own launches {on}, {at}, {k}")
        m.close()


@BOTH
@pytest.mark.parametrize("rows,beside", [(4096, True), (4097, False)])
def test_most_keys(gpu, dtype, rows, beside):
    """The route goes by the most keys that a position can see, at its border: three launches a layer or five."""
    kw = dict(heads=4, kv_heads=1, dim=64, vdim=64)
    mod = U.Model(U.gusorax([U.chunked(chunk=5000, **kw)], positions=5000))
    m = mod.load(dtype, max_seq_len=rows)
    assert m.cfg.launches_per_token == (5 if beside else 7)
    toks = mod.tokens(140)
    U.check(U.run_alone(m, toks, tuple(range(130, 140))), mod.logits(toks), dtype, "steps")
    m.close()


@pytest.mark.parametrize("heads,kv_heads,dtype,keys,most", [
    (8, 8, "bfloat16", 4096, 4096), (9, 9, "bfloat16", 1024, 1024), (9, 9, "float32", 2048, 2048), (36, 4, "bfloat16", 1024, 1024),
    (33, 33, "float32", 512, 512), (33, 33, "bfloat16", 256, 256), (65, 65, "float32", 256, 256), (130, 65, "bfloat16", 128, 128)])
def test_more_groups_than_splits_for_them(gpu, heads, kv_heads, dtype, keys, most):
    """The bound follows the splits, which many groups of heads share: at the bound beside the experts, above it as launches of
    their own; steps up to it, and behind a window that has moved on."""
    for window, launches in ((keys, 5), (keys + 1, 7)):
        kw = dict(heads=heads, kv_heads=kv_heads, dim=6, vdim=5)
        mod = U.Model(U.gusorax([dict(U.windowed(window=window, rows=8, far=60.0, **kw), mlp=U.clamped())], positions=4400))
        m = mod.load(dtype, max_seq_len=min(max(2 * most, 300), 4400), max_seqs=4)
        assert m.cfg.launches_per_token == launches
        if most <= 512:
            toks = mod.tokens(most + 40)
            want = mod.logits(toks)
            for at in ([most - 3], [0, 30, most // 2, most + 20]):
                for k, g in zip(at, steps(m, toks, at, 6)):
                    U.check(g, want[k: k + 6], dtype, f"{window} {at} {k}")
        m.close()


def test_fences_give_the_same_bits(gpu):
    """The hand-over of the splits with release and acquire fences and without, many steps beside a stream of experts."""
    mod = U.Model(U.gusorax([dict(U.windowed(heads=8, kv_heads=2, dim=128, vdim=128, window=400, rows=16, far=90.0),
                                  mlp=U.clamped(16, 6, 512))] * 3, width=512))
    toks = mod.tokens(380)
    out = []
    for fenced in (None, "1"):
        _ffi.debug_set("KH_ATTN_FENCED", fenced)
        try:
            m = mod.load("float32", max_seqs=4)
        finally:
            _ffi.debug_set("KH_ATTN_FENCED", None)
        out.append([steps(m, toks, [300, 40, 129, 5], 64) for _ in range(3)])
        m.close()
    for got in out[0] + out[1]:
        np.testing.assert_array_equal(got, out[1][0])


@BOTH
def test_hand_over_is_checked_at_creation(gpu, dtype):
    """Splits merged without fences against the fenced form, on the model's own device: the result in the configuration, the fenced
    form where the check fails (injected), nothing where no launch has several splits."""
    kw = dict(heads=8, kv_heads=2, dim=128, vdim=64)
    mod = U.Model(U.gusorax([dict(U.chunked(), mlp=U.dense()), dict(U.windowed(window=400, rows=16, far=90.0, **kw), mlp=U.clamped())]))
    toks = mod.tokens(310)
    out = {}
    for hooks, want in (((), 1), ((("KH_SELFTEST_FAIL", "attn"),), -1), ((("KH_SELFTEST", "0"),), 0), ((("KH_ATTN_FENCED", "1"),), 2)):
        for k, v in hooks:
            _ffi.debug_set(k, v)
        try:
            m = mod.load(dtype, max_seqs=4)
        finally:
            for k, _ in hooks:
                _ffi.debug_set(k, None)
        assert m.cfg.attn_merge_selftest == want and m.cfg.ring_selftest == 0
        out[want] = steps(m, toks, [300, 0, 63, 64], 6)
        m.close()
    U.check(out[1][0], mod.logits(toks)[300:306], dtype)
    for v in out.values():
        np.testing.assert_array_equal(v, out[1])
    split = 32 if dtype == "float32" else 64
    for layer, rows, want in ((U.windowed(window=split, **kw), 512, 0), (U.windowed(window=split + 1, **kw), 512, 1),
                              (U.chunked(chunk=300, **kw), split, 0), (U.latent(), 512, 0)):
        one = U.Model(U.config([layer]) if layer["type"] == "latent_attention" else U.gusorax([dict(layer, mlp=U.dense())]))
        m = one.load(dtype, max_seq_len=rows)
        assert m.cfg.attn_merge_selftest == want, (layer, rows)
        m.close()
