"""Prompt passes on pairs of halves (csrc/kh_pair.h) against 64 bits, with weights whose sizes differ by powers of two that
cancel over two matrices: the rows are held to the error of the fp32 matrix cores on the same weights (KH_PG_PAIR=0)."""
import dataclasses

import numpy as np
import pytest
import torch

import exact_kv
from kuiperllama_amd import _ffi, binfmt
from test_model_gpu import _PF_SPECS

pytestmark = pytest.mark.gpu


def _scale(t, name, index, f, axis):
    """Rows (axis 0) or columns (axis 1) of a matrix times f; int8 matrices: the scales of the 64-column groups."""
    w = t[name]
    if w.dtype != torch.int8:
        if axis == 0:
            w[index] *= f
        else:
            w[:, index] *= f
        return
    s = t[name + ".scales"].reshape(w.shape[0], -1)
    if axis == 0:
        s[index] *= f
    else:
        s[:, index // 64] *= f


def _gated_unit(t, l, spec, f):  # one row of w1, another one of w3
    _scale(t, f"w1.{l}", 5, f, 0)
    _scale(t, f"w3.{l}", 700, f, 0)
    _scale(t, f"w2.{l}", 5, 1 / f, 1)
    _scale(t, f"w2.{l}", 700, 1 / f, 1)


def _up(t, l, spec, f):  # one row of w3
    _scale(t, f"w3.{l}", 700, f, 0)
    _scale(t, f"w2.{l}", 700, 1 / f, 1)


def _norms(t, l, spec, f):  # one weight of either norm
    for n, mats in (("att_norm", ("wq", "wk", "wv")), ("ffn_norm", ("w1", "w3"))):
        t[f"{n}.{l}"][70:71] *= f
        for k in mats:
            _scale(t, f"{k}.{l}", 70, 1 / f, 1)


def _values(t, l, spec, f):  # one value column of a head
    g, d = spec.n_kv_heads - 1, 3
    _scale(t, f"wv.{l}", g * spec.head_size + d, f, 0)
    for h in range(g * spec.kv_mul, (g + 1) * spec.kv_mul):
        _scale(t, f"wo.{l}", h * spec.head_size + d, 1 / f, 1)


def errors(monkeypatch, img, spec, n, hook="KH_PG_PAIR", front=None):
    """Error of the rows of the layers behind the first: with pairs, and with `hook` off.  front: cache rows before them."""
    from kuiperllama_amd.model import KuiperModel
    toks = [int(t) for t in np.random.default_rng(17).integers(0, spec.vocab_size, n)]
    want = exact_kv.rows(img, spec, toks, front)
    old = 0 if front is None else len(front[0][0])
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv(hook, "0")
        m = KuiperModel.from_device_image(img, spec)
        for l in range(spec.n_layers if old else 0):
            m.write_kv(l, 0, *front[l])
        m.prefill_gemm(toks, old)
        got = [m.read_kv(l, old, n) for l in range(1, spec.n_layers)]
        out.append(max(exact_kv.error(g, w) for a, b in zip(got, want[1:]) for g, w in zip(a, b)))
        m.close()
        monkeypatch.delenv(hook, raising=False)
    return out


@pytest.mark.parametrize("change", [_gated_unit, _up, _norms])
@pytest.mark.parametrize("name", ["gqa-half", "mha-interleaved", "int8"])
@pytest.mark.parametrize("e", [0, 6, 12, 15])
@pytest.mark.parametrize("n", [30, 150])  # the gated unit with a scale per 32 and per 64 columns
def test_sizes_that_cancel(gpu, name, change, e, n, monkeypatch):
    spec = _PF_SPECS[name]
    img = binfmt.synth_image(spec, seed=51, device=gpu)
    t = exact_kv.tensors(img, spec)
    for l in range(spec.n_layers):
        change(t, l, spec, 2.0 ** e)
    pair, fp32 = errors(monkeypatch, img, spec, n)
    print(f"{name} {change.__name__} 2^{e}, {n} tokens: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32  # a quarter for the luck of the roundings


@pytest.mark.parametrize("name", ["gqa-half", "mha-interleaved", "gqa-half-hs128", "int8"])
@pytest.mark.parametrize("e", [0, 6, 12, 15])
def test_value_columns_that_cancel(gpu, name, e, monkeypatch):
    """Attention of a slice on pairs (csrc/kh_pattn_pair.h) against the fp32 matrix cores."""
    spec = _PF_SPECS[name]
    img = binfmt.synth_image(spec, seed=52, device=gpu)
    t = exact_kv.tensors(img, spec)
    for l in range(spec.n_layers):
        _values(t, l, spec, 2.0 ** e)
    pair, fp32 = errors(monkeypatch, img, spec, 300, "KH_PAIR_ATTN")
    print(f"{name} values 2^{e}: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32


@pytest.mark.parametrize("name", ["gqa-half", "gqa-half-hs128"])
def test_rows_of_the_caller_in_front(gpu, name, monkeypatch):
    """Cache rows that the model cannot have computed: values of 1e4, keys a thousandth of the usual ones."""
    spec = _PF_SPECS[name]
    img = binfmt.synth_image(spec, seed=53, device=gpu)
    rng = np.random.default_rng(18)
    draw = lambda size: (size * rng.standard_normal((70, spec.kv_dim))).astype(np.float32)
    front = [(draw(1e-3), draw(1e4)) for _ in range(spec.n_layers)]
    pair, fp32 = errors(monkeypatch, img, spec, 250, "KH_PAIR_ATTN", front)
    print(f"{name} rows in front: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32


def test_rows_handed_back_change_nothing(gpu):
    """A caller that reads rows and writes them back gets the same rows behind them: the pass does not depend on who wrote
    the cache."""
    from kuiperllama_amd.model import KuiperModel
    spec = _PF_SPECS["gqa-half"]
    img = binfmt.synth_image(spec, seed=54, device=gpu)
    toks = [int(t) for t in np.random.default_rng(19).integers(0, spec.vocab_size, 400)]
    out = []
    for back in (False, True):
        m = KuiperModel.from_device_image(img, spec)
        m.prefill_gemm(toks[:100], 0)
        for l in range(spec.n_layers if back else 0):
            m.write_kv(l, 0, *m.read_kv(l, 0, 100))
        m.prefill_gemm(toks[100:], 100)
        out.append([m.read_kv(l, 100, 300) for l in range(spec.n_layers)])
        m.close()
    for a, b in zip(*out):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("shape", [None, "0,1", "1,4", "2,2", "3,4"])
@pytest.mark.parametrize("first", [0.0, 2.0 ** -24, 2.0 ** 10])
def test_first_columns_of_another_size(gpu, first, shape, monkeypatch):
    """The scale of a weight row comes from its first 32 columns: rows where these (and those in front of a K slice) are zero,
    tiny or large.  Large ones meet inputs as much smaller."""
    spec = _PF_SPECS["gqa-half"]
    img = binfmt.synth_image(spec, seed=55, device=gpu)
    t = exact_kv.tensors(img, spec)
    for l in range(spec.n_layers):
        for n, norm in (("wq", "att_norm"), ("wk", "att_norm"), ("wv", "att_norm"), ("w1", "ffn_norm"), ("w3", "ffn_norm"),
                        ("wo", None), ("w2", None)):
            w = t[f"{n}.{l}"]
            if first > 1 and norm is None:
                continue
            w[::3, :32] *= first
            if norm is None:
                w[::3, w.shape[1] // 2: w.shape[1] // 2 + 32] *= first
        if first > 1:
            for norm in ("att_norm", "ffn_norm"):
                t[f"{norm}.{l}"][:32] /= first
    if shape:
        monkeypatch.setenv("KH_PAIR_SHAPE", shape)
    pair, fp32 = errors(monkeypatch, img, spec, 150)
    print(f"first columns {first:.2g}, shape {shape}: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32


@pytest.mark.parametrize("name", ["gqa-half", "qwen-bias", "int8"])
def test_weights_written_in_place(gpu, name):
    """Weights that the caller owns may be written between two calls: the rows are those of a model made afterwards."""
    from kuiperllama_amd.model import KuiperModel
    spec = _PF_SPECS[name]
    img = binfmt.synth_image(spec, seed=56, device=gpu)
    toks = [int(t) for t in np.random.default_rng(20).integers(0, spec.vocab_size, 300)]
    m = KuiperModel.from_device_image(img, spec)
    m.prefill_gemm(toks, 0)
    for e in binfmt.layout(spec)[0]:
        w = binfmt.tensor_from_image(img, e)
        base = e.name.split(".")[0]
        if e.name.endswith("scales") or (w.dtype == torch.float32 and base[0] in "wb"):
            k = torch.arange(w.numel(), device=gpu).reshape(w.shape) // w.shape[-1] % 3
            w.mul_(torch.where(k == 0, 64.0, 1 / 64.0))
    torch.cuda.synchronize()
    m.prefill_gemm(toks, 0)
    fresh = KuiperModel.from_device_image(img, spec)
    fresh.prefill_gemm(toks, 0)
    for l in range(spec.n_layers):
        for a, b in zip(m.read_kv(l, 0, 300), fresh.read_kv(l, 0, 300)):
            assert np.isfinite(a).all() and np.array_equal(a, b), l
    m.close()
    fresh.close()


def test_uneven_rows_cost_a_second_pass(gpu):
    """Rows with one number far above their first 32 columns: the waves that meet them compute their tiles a second time
    behind a search for the scales: 1.9 to 2.2 times the time of even rows; 3.3 with one request in flight."""
    from kuiperllama_amd.model import KuiperModel
    spec = dataclasses.replace(binfmt.PRESETS["llama3.2-1b"], n_layers=3, vocab_size=2000, seq_len=1024)
    toks = [int(t) for t in np.random.default_rng(25).integers(0, spec.vocab_size, 512)]
    ms = []
    for uneven in (False, True):
        img = binfmt.synth_image(spec, seed=60, device=gpu)
        t = exact_kv.tensors(img, spec)
        for l in range(spec.n_layers if uneven else 0):
            for n in ("wq", "wk", "wv", "wo", "w1", "w3", "w2"):
                w = t[f"{n}.{l}"]
                w[7::100, 1000] = 200 * w.abs().max()
        m = KuiperModel.from_device_image(img, spec)
        m.time_prefill(toks, 0)
        ms.append(min(m.time_prefill(toks, 0) for _ in range(8)))
        m.close()
    print(f"{ms[0]:.3f} ms, with uneven rows {ms[1]:.3f}")
    assert ms[1] < 2.6 * ms[0]


_WIDTHS = {
    # 480 = 7.5 groups of 64 columns, heads of 96 (attention outputs through k_pair_convert), hidden 1376 = 21.5 groups
    "odd": binfmt.ModelSpec(480, 1376, 2, 5, 5, 500, 512, True, binfmt.FAMILY_LLAMA, False, 64, binfmt.ROPE_HALF, 10000.0, 1e-5, "odd"),
    # rows that k_pair_rmsnorm does not keep in registers
    "wide": binfmt.ModelSpec(4608, 512, 2, 36, 4, 500, 512, True, binfmt.FAMILY_LLAMA, False, 64, binfmt.ROPE_INTERLEAVED, 10000.0,
                             1e-5, "wide"),
}


@pytest.mark.parametrize("name", sorted(_WIDTHS))
@pytest.mark.parametrize("n", [3, 70, 300])
def test_widths(gpu, name, n, monkeypatch):
    spec = _WIDTHS[name]
    img = binfmt.synth_image(spec, seed=57, device=gpu)
    pair, fp32 = errors(monkeypatch, img, spec, n)
    print(f"{name}, {n} tokens: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32


_SLICES = {
    # wo in four slices: the second begins at stage 14 of the 16 whose scales travel together (Qwen2.5-0.5B up to 128 tokens)
    "fp32": (binfmt.ModelSpec(896, 1792, 2, 14, 2, 500, 512, True, binfmt.FAMILY_LLAMA, False, 64, binfmt.ROPE_HALF, 10000.0, 1e-5,
                              "slices"), None),
    # w2 in four slices that begin at stages 15, 31 and 47
    "int8": (binfmt.ModelSpec(512, 4032, 2, 8, 2, 500, 512, False, binfmt.FAMILY_LLAMA, True, 64, binfmt.ROPE_HALF, 10000.0, 1e-5,
                              "slices8"), "2,4"),
}


@pytest.mark.parametrize("name", sorted(_SLICES))
@pytest.mark.parametrize("n", [16, 41, 128])
def test_slices_that_begin_behind_the_first_scales(gpu, name, n, monkeypatch):
    """A K slice whose second stages need the next 16 scales: those have landed too."""
    spec, shape = _SLICES[name]
    if shape:
        monkeypatch.setenv("KH_PAIR_SHAPE", shape)
    else:
        plan = _ffi.plan_pair_shapes(spec.dim, spec.hidden_dim, spec.kv_dim, False, n)["wo"]
        assert (plan["bm"], plan["bn"], plan["kz"]) == (32, 64, 4)
    img = binfmt.synth_image(spec, seed=59, device=gpu)
    pair, fp32 = errors(monkeypatch, img, spec, n)
    print(f"{name}, {n} tokens: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_token_that_is_not_finite(gpu, bad):
    """An embedding row that is not finite spoils its own position and those behind it: blocks of positions in front of it
    stay within the error of the rest (the waves that meet it compute their tiles a second way)."""
    from kuiperllama_amd.model import KuiperModel
    spec = _PF_SPECS["gqa-half"]
    img = binfmt.synth_image(spec, seed=58, device=gpu)
    toks = [int(t) for t in np.random.default_rng(24).integers(0, spec.vocab_size - 1, 300)]
    toks[200] = spec.vocab_size - 1
    want = exact_kv.rows(img, spec, toks[:192])
    exact_kv.tensors(img, spec)["tok_emb"][spec.vocab_size - 1, 17] = bad
    m = KuiperModel.from_device_image(img, spec)
    m.prefill_gemm(toks, 0)
    for l in range(spec.n_layers):
        for got, w in zip(m.read_kv(l, 0, 192), want[l]):
            assert exact_kv.error(got, w) < 2e-6, l  # 1.2e-6: the largest on the fp32 matrix cores without it
        assert not np.isfinite(m.read_kv(l, 200, 1)[0]).all()
    m.close()
