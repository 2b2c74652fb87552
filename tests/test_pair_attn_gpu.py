"""Attention of a prompt slice with pairs of halves (csrc/kh_pattn_pair.h) against the fp32 matrix cores (KH_PAIR_ATTN=0),
which the oracle tests hold: edges of the 16-token tiles and 32-position blocks, blocks per wave, the line of the dispatch."""
import numpy as np
import pytest
import torch

from kuiperllama_amd import binfmt
from test_model_gpu import KV_ATOL_GEMM

pytestmark = pytest.mark.gpu


def _spec(hs, heads, kv_heads, half):
    return binfmt.ModelSpec(hs * heads, 512, 2, heads, kv_heads, 500, 1024, True, binfmt.FAMILY_LLAMA, False, 64,
                            binfmt.ROPE_HALF if half else binfmt.ROPE_INTERLEAVED, 10000.0, 1e-5, f"pair-attn-{hs}")


def _both(monkeypatch, img, spec, slices):
    from kuiperllama_amd.model import KuiperModel
    out = []
    for hook in (None, "0"):
        if hook:
            monkeypatch.setenv("KH_PAIR_ATTN", hook)
        m = KuiperModel.from_device_image(img, spec)
        for toks, pos in slices:
            m.prefill_gemm(toks, pos)
        out.append(m.read_kv(1, 0, slices[-1][1] + len(slices[-1][0])))  # layer 1 sees the attention of layer 0
        m.close()
        monkeypatch.delenv("KH_PAIR_ATTN", raising=False)
    return out


GEOMETRIES = [(48, 6, 6, False), (64, 8, 2, True), (64, 4, 4, False), (128, 4, 1, True), (128, 2, 2, False)]


@pytest.mark.parametrize("hs,heads,kv_heads,half", GEOMETRIES)
def test_slices(gpu, hs, heads, kv_heads, half, monkeypatch):
    spec = _spec(hs, heads, kv_heads, half)
    img = binfmt.synth_image(spec, seed=41, device=gpu)
    toks = [int(t) for t in np.random.default_rng(8).integers(0, spec.vocab_size, 1024)]
    cases = [[(toks[:n], 0)] for n in (255, 256, 257, 271, 273, 288, 289, 511, 513, 1000)]
    cases += [[(toks[:p], 0), (toks[p:p + n], p)] for p, n in ((193, 127), (193, 128), (224, 129), (300, 161), (511, 400), (512, 512))]
    for slices in cases:
        a, b = _both(monkeypatch, img, spec, slices)
        for x, y in zip(a, b):  # either is within KV_ATOL_GEMM of the oracle's rows
            np.testing.assert_allclose(x, y, rtol=0, atol=2 * KV_ATOL_GEMM, err_msg=str([(len(t), p) for t, p in slices]))


@pytest.mark.parametrize("hs,heads,kv_heads,half", GEOMETRIES[1:4])
def test_spread_of_values_and_scores(gpu, hs, heads, kv_heads, half, monkeypatch):
    """Value rows between 2^-20 and 1 of their usual size, some zero; queries 16 times as large, so that a few positions
    carry a row.  An fp32 score of size s has an error of s 2^-24 per rounding, here s < 2^8 and some 2^3 roundings: the
    weights, and with them the rows, move by 2^-13 at most between two orders of summation.  Columns far below the row's
    largest entry are held by test_pair_exact_gpu.py."""
    spec = _spec(hs, heads, kv_heads, half)
    img = binfmt.synth_image(spec, seed=42, device=gpu)
    for e in binfmt.layout(spec)[0]:
        base = e.name.split(".")[0]
        if base == "wv":
            w = binfmt.tensor_from_image(img, e)
            k = torch.arange(e.shape[0], device=gpu) % 21
            w.copy_(w * torch.exp2(-k.float())[:, None])
            w[1].zero_()
        elif base == "wq":
            w = binfmt.tensor_from_image(img, e)
            w.copy_(w * 16)
    _close(monkeypatch, img, spec)


@pytest.mark.parametrize("exp", [-30, -70, -90])
def test_tiny_queries_and_keys(gpu, exp, monkeypatch):
    """Scales of a block and of a token whose product leaves the range of fp32: every score is zero, masked ones stay masked."""
    spec = _spec(64, 8, 2, True)
    img = binfmt.synth_image(spec, seed=43, device=gpu)
    for e in binfmt.layout(spec)[0]:
        if e.name.split(".")[0] in ("wq", "wk"):
            w = binfmt.tensor_from_image(img, e)
            w.copy_(w * 2.0 ** exp)
    _close(monkeypatch, img, spec)


def _close(monkeypatch, img, spec):
    toks = [int(t) for t in np.random.default_rng(9).integers(0, spec.vocab_size, 600)]
    a, b = _both(monkeypatch, img, spec, [(toks, 0)])
    for x, y in zip(a, b):
        assert np.isfinite(x).all()
        top = np.abs(y).max(axis=1, keepdims=True)
        assert (np.abs(x - y) / top).max() < 2.0 ** -13, float((np.abs(x - y) / top).max())
