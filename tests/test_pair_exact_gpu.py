"""Prompt passes on pairs of halves (csrc/kh_pair.h) against 64 bits, with weights whose sizes differ by powers of two that
cancel over two matrices: the rows are held to the error of the fp32 matrix cores on the same weights (KH_PG_PAIR=0)."""
import numpy as np
import pytest
import torch

import exact_kv
from kuiperllama_amd import binfmt
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


def errors(monkeypatch, img, spec, n, hook="KH_PG_PAIR", pos=0):
    """Error of the rows of the layers behind the first: with pairs, and with `hook` off."""
    from kuiperllama_amd.model import KuiperModel
    toks = [int(t) for t in np.random.default_rng(17).integers(0, spec.vocab_size, n)]
    want = exact_kv.rows(img, spec, toks)
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv(hook, "0")
        m = KuiperModel.from_device_image(img, spec)
        m.prefill_gemm(toks, 0)
        got = [m.read_kv(l, 0, n) for l in range(1, spec.n_layers)]
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
