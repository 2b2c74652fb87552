"""Attention and wo of a decoded token in one launch (csrc/kh_attn_wo.h): positions at the edges of its 16-timestep tiles, of
its two tiles a wave and of its range, and every shape of its rows."""
import numpy as np
import pytest
import torch

from kuiperllama_amd import binfmt

pytestmark = pytest.mark.gpu


def _spec(dim, hidden, heads, kv, name):
    return binfmt.ModelSpec(dim, hidden, 2, heads, kv, 700, 512, True, binfmt.FAMILY_LLAMA, False, 64, binfmt.ROPE_HALF, 500000.0,
                            1e-5, name)


# head size 48: 16 and 32 lanes a row (stories15M's; two heads a group); 64: one float4 a lane (32 lanes, 64 lanes), two of them,
# of which the second is half empty (seven heads), one and two rows, rows past the end of the last slice (dim 896, 1088)
_SPECS = {s.name: s for s in (
    _spec(288, 768, 6, 6, "48x6-6"), _spec(384, 768, 8, 4, "48x8-4"), _spec(512, 1408, 8, 4, "64x8-4"),
    _spec(448, 1216, 7, 1, "64x7-1"), _spec(768, 2112, 12, 6, "64x12-6"), _spec(896, 1216, 14, 2, "64x14-2"), _spec(1024, 1408, 16, 8, "64x16-8"),
    _spec(1088, 1408, 17, 1, "64x17-1"),  # seventeen heads a group: the launches of their own
    _spec(2048, 1408, 32, 8, "64x32-8"), _spec(2048, 1408, 32, 4, "64x32-4"))}


@pytest.mark.parametrize("name,hook,per", [("48x6-6", None, 4), ("64x32-8", None, 4), ("64x17-1", None, 5), ("64x32-8", "0", 5)])
def test_launches_per_token(gpu, name, hook, per, monkeypatch):
    """The count that the configuration reports is that of the step at position 0."""
    from kuiperllama_amd.model import KuiperModel
    if hook:
        monkeypatch.setenv("KH_ATTN_WO", hook)
    spec = _SPECS[name]
    m = KuiperModel.from_device_image(binfmt.synth_image(spec, seed=31, device=gpu), spec)
    assert m.cfg.launches_per_token == per * spec.n_layers + 2
    assert sum(v["launches_per_step"] for v in m.profile_step(0, 1).values()) == m.cfg.launches_per_token
    m.close()


@pytest.mark.parametrize("heads,kv,joint", [(32, 8, True), (35, 7, False), (36, 6, False), (40, 8, False)])
def test_wide_models_with_wide_workgroups(gpu, heads, kv, joint, monkeypatch):
    """With 512 threads in ffn13 two float4 a thread cover 4096 columns; eight prompt tokens of more than 2048 do not fit the LDS of
    the joint form's prompt launch, so such models keep their launches apart."""
    from kuiperllama_amd.model import KuiperModel
    monkeypatch.setenv("KH_SHAPE_FFN", "1,8,256,512")
    spec = _spec(64 * heads, 1408, heads, kv, "wide")
    img = binfmt.synth_image(spec, seed=31, device=gpu)
    a, b = KuiperModel.from_device_image(img, spec), KuiperModel.from_device_image(img, spec)
    assert a.cfg.launches_per_token == (4 if joint else 5) * spec.n_layers + 2
    toks = [int(t) for t in np.random.default_rng(4).integers(0, spec.vocab_size, 21)]
    a.prefill(toks, 0)
    for pos, t in enumerate(toks):
        b.predict(t, pos, exec="fused")
    for l in range(spec.n_layers):
        for x, y in zip(a.read_kv(l, 0, len(toks)), b.read_kv(l, 0, len(toks))):
            np.testing.assert_array_equal(x, y)
    a.close()
    b.close()


def test_profiles_name_what_is_launched(gpu):
    """Below the end of their range attention and wo are one launch and are reported as one; behind it each has its own time."""
    from kuiperllama_amd import _ffi
    from kuiperllama_amd.model import KuiperModel
    spec = _SPECS["64x12-6"]
    end = _ffi.plan_attn_wo(spec.dim, spec.hidden_dim, spec.n_heads, spec.n_kv_heads, spec.seq_len)["end"]
    assert end == 192
    m = KuiperModel.from_device_image(binfmt.synth_image(spec, seed=31, device=gpu), spec)
    m.generate([1, 2], 300)
    joint, apart = ["qkv", "attn_wo", "ffn13", "w2", "cls", "sample"], ["qkv", "attn", "wo", "ffn13", "w2", "cls", "sample"]
    for pos, names in ((0, joint), (64, joint), (end - 1, joint), (end, apart), (290, apart)):
        us = m.profile_kernels(pos)
        assert sorted(us) == sorted(names) and min(us.values()) > 0.5, (pos, us)
        if names is joint:
            with pytest.raises(_ffi.KhError) as e:
                m.profile_kernel("wo", pos)
            assert e.value.code == _ffi.KH_ERR_UNSUPPORTED
            assert m.profile_kernel("attn", pos) > 0.5
        else:
            assert m.profile_kernel("wo", pos) > 0.5
        step = m.profile_step(pos, 1)
        assert sorted(step) == sorted(names)
        for k, v in step.items():
            assert v["launches_per_step"] == (1 if k in ("cls", "sample") else spec.n_layers) and v["avg_us"] > 0.5, (pos, k, v)
    m.close()


@pytest.mark.parametrize("name", ["48x6-6", "64x8-4", "64x32-8"])
def test_launches_of_their_own(gpu, oracle, name, monkeypatch):
    """The same models with attention and wo apart at every position: the oracle's logits, and the prompt path's bits."""
    from kuiperllama_amd.model import KuiperModel
    monkeypatch.setenv("KH_ATTN_WO", "0")
    spec = _SPECS[name]
    img_d = binfmt.synth_image(spec, seed=31, device=gpu, final_norm_std=1.0)
    torch.cuda.synchronize()
    a, b = KuiperModel.from_device_image(img_d, spec), KuiperModel.from_device_image(img_d, spec)
    om = oracle.OracleModel.from_spec(img_d.cpu().numpy(), spec)
    toks = [int(t) for t in np.random.default_rng(5).integers(0, spec.vocab_size, 140)]
    for pos, t in enumerate(toks):
        a.predict(t, pos, exec="fused")
        want = om.forward(t, pos)
        if pos in (0, 1, 15, 16, 63, 127, 128, 139):
            err = np.abs(a.logits() - want).max()
            assert err <= 4e-5, f"position {pos}: {err:.3e}"
    b.prefill(toks[:-1], 0)
    b.predict(toks[-1], 139, exec="fused")
    assert np.array_equal(a.logits(), b.logits())
    a.close()
    b.close()


@pytest.mark.parametrize("name,pos0,n", [("64x12-6", 4, 300), ("64x12-6", 187, 9), ("64x12-6", 0, 197), ("64x32-8", 251, 9)])
def test_token_by_token_prompt_across_the_end(gpu, name, pos0, n):
    """The prompt phase one token a step leaves the cache rows of predict() at every position, whatever its first one is: no graph
    of several steps crosses the end of the range, 192 or 256."""
    from kuiperllama_amd.model import KuiperModel
    spec = _SPECS[name]
    img = binfmt.synth_image(spec, seed=31, device=gpu, final_norm_std=1.0)
    a, b = KuiperModel.from_device_image(img, spec), KuiperModel.from_device_image(img, spec)
    toks = [int(t) for t in np.random.default_rng(4).integers(0, spec.vocab_size, pos0 + n)]
    for pos, t in enumerate(toks):
        a.predict(t, pos, exec="fused")
        if pos < pos0:
            b.predict(t, pos, exec="fused")
    assert b.time_prefill(toks[pos0:], pos0, "token") > 0
    for l in range(spec.n_layers):
        for x, y in zip(a.read_kv(l, 0, pos0 + n), b.read_kv(l, 0, pos0 + n)):
            np.testing.assert_array_equal(x, y)
    a.close()
    b.close()


@pytest.mark.parametrize("heads,kv,end", [(12, 6, 192), (10, 5, 128), (21, 7, 64), (14, 2, 256)])
def test_bits_follow_from_the_position(gpu, heads, kv, end):
    """Steps, graphs of several and the prompt path of several tokens across an end of the range that is not 256."""
    from kuiperllama_amd import _ffi
    from kuiperllama_amd.model import KuiperModel
    spec = _spec(64 * heads, 1408, heads, kv, "end")
    assert _ffi.plan_attn_wo(spec.dim, 1408, heads, kv, spec.seq_len)["end"] == end
    img = binfmt.synth_image(spec, seed=31, device=gpu, final_norm_std=1.0)
    a, b = KuiperModel.from_device_image(img, spec), KuiperModel.from_device_image(img, spec)
    toks = [int(t) for t in np.random.default_rng(6).integers(0, spec.vocab_size, end + 11)]
    for pos, t in enumerate(toks):
        a.predict(t, pos, exec="fused")
    b.prefill(toks[:-1], 0)
    b.predict(toks[-1], len(toks) - 1, exec="fused")
    for l in range(spec.n_layers):
        for x, y in zip(a.read_kv(l, 0, len(toks)), b.read_kv(l, 0, len(toks))):
            np.testing.assert_array_equal(x, y)
    assert np.array_equal(a.logits(), b.logits())
    words, _ = a.generate(toks[:3], end + 21, exec="graph")
    assert words == b.generate(toks[:3], end + 21, exec="fused")[0]
    assert np.array_equal(a.logits(), b.logits())
    a.close()
    b.close()


@pytest.mark.parametrize("name", sorted(_SPECS))
def test_against_the_oracle_and_the_prompt_path(gpu, oracle, name, monkeypatch):
    """Logits within the bound of fp32 decode steps (4e-5, as for the attention in launches of its own); the prompt path of
    several tokens a weight pass leaves the same bits, also where a chunk would cross the end of the range; words of captured and
    eager steps are the same across it."""
    from kuiperllama_amd.model import KuiperModel
    monkeypatch.setenv("KH_ATTN_WO", "256")  # the whole range that the kernels have, wherever they pay
    spec = _SPECS[name]
    img_d = binfmt.synth_image(spec, seed=31, device=gpu, final_norm_std=1.0)  # words that wander
    torch.cuda.synchronize()
    img_h = img_d.cpu().numpy()
    a, b = KuiperModel.from_device_image(img_d, spec), KuiperModel.from_device_image(img_d, spec)
    om = oracle.OracleModel.from_spec(img_h, spec)
    ko, vo = om.kv_cache()
    rng = np.random.default_rng(3)
    for l in range(spec.n_layers):
        k, v = (rng.standard_normal((300, spec.kv_dim), dtype=np.float32) for _ in range(2))
        k[rng.integers(0, 300, 6)] *= 6.0  # a few dominant keys: the waves' maxima differ
        ko[l, :300], vo[l, :300] = k, v
        a.write_kv(l, 0, k, v)
        b.write_kv(l, 0, k, v)
    for pos in (0, 1, 15, 16, 63, 127, 128, 143, 254, 255, 256):
        tok = int(rng.integers(0, spec.vocab_size))
        a.predict(tok, pos, exec="fused")
        b.predict(tok, pos, exec="fused")
        err = np.abs(a.logits() - om.forward(tok, pos)).max()
        assert err <= 4e-5, f"position {pos}: {err:.3e}"
    toks = [int(t) for t in rng.integers(0, spec.vocab_size, 24)]
    a.prefill(toks[:-1], 240)  # 240 .. 262
    for i, t in enumerate(toks):
        b.predict(t, 240 + i, exec="fused")
    a.predict(toks[-1], 263, exec="fused")
    for l in range(spec.n_layers):
        for x, y in zip(a.read_kv(l, 0, 264), b.read_kv(l, 0, 264)):
            assert np.array_equal(x, y), l
    assert np.array_equal(a.logits(), b.logits())
    words, _ = a.generate(toks[:3], 270, exec="graph")
    assert words == b.generate(toks[:3], 270, exec="fused")[0]
    assert np.array_equal(a.logits(), b.logits())
    a.close()
    b.close()
