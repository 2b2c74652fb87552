"""Pair GEMMs of the prompt phase (csrc/kh_pair.h): every tile and K split at the edges of its token and row tiles, and
the scales, against the fp32-MFMA GEMMs of the same pass (KH_PG_PAIR=0), which the oracle tests hold."""
import dataclasses

import numpy as np
import pytest
import torch

from kuiperllama_amd import binfmt
from test_model_gpu import _PF_SPECS, KV_ATOL_GEMM

pytestmark = pytest.mark.gpu

SPECS = dict(_PF_SPECS)
# 48 heads of 48: a head is no multiple of 32 rows; 288 = 9 blocks of 32: an odd number of stages, 2.25 row tiles of 128
SPECS["stories"] = binfmt.ModelSpec(288, 768, 2, 6, 6, 500, 512, True, binfmt.FAMILY_LLAMA, False, 64,
                                    binfmt.ROPE_INTERLEAVED, 10000.0, 1e-5, "pair-stories")


def _rows(m, n):
    return [np.concatenate(m.read_kv(l, 0, n), 1) for l in range(m.cfg.layer_num)]


def _both(monkeypatch, img, spec, run, n):
    from kuiperllama_amd.model import KuiperModel
    out = []
    for pair in (None, "0"):
        if pair:
            monkeypatch.setenv("KH_PG_PAIR", pair)
            monkeypatch.delenv("KH_PAIR_SHAPE", raising=False)
        m = KuiperModel.from_device_image(img, spec)
        run(m)
        out.append(_rows(m, n))
        m.close()
        monkeypatch.delenv("KH_PG_PAIR", raising=False)
    return out


@pytest.mark.parametrize("name", sorted(SPECS))
@pytest.mark.parametrize("shape", [None, "0,1", "0,4", "1,2", "2,1", "2,4", "3,2"])
def test_tiles_and_splits(gpu, name, shape, monkeypatch):
    spec = dataclasses.replace(SPECS[name], seq_len=1024)
    img = binfmt.synth_image(spec, seed=31, device=gpu)
    toks = [int(t) for t in np.random.default_rng(5).integers(0, spec.vocab_size, 900)]
    atol = 2 * KV_ATOL_GEMM * (4 if spec.quant else 1)  # either path is within KV_ATOL_GEMM of the oracle's rows
    for n in (1, 31, 33, 63, 65, 111, 113, 127, 129, 225, 800):
        if shape:
            monkeypatch.setenv("KH_PAIR_SHAPE", shape)
        a, b = _both(monkeypatch, img, spec, lambda m: m.prefill_gemm(toks[:n], 0), n)
        for l, (x, y) in enumerate(zip(a, b)):
            np.testing.assert_allclose(x, y, rtol=0, atol=atol, err_msg=f"{name} {shape} n={n} layer {l}")


@pytest.mark.parametrize("name", ["gqa-half", "int8"])
def test_long_pass_and_second_pass(gpu, name, monkeypatch):
    """2048 tokens in one pass, then a remainder at position 2048."""
    spec = dataclasses.replace(SPECS[name], seq_len=2304)
    img = binfmt.synth_image(spec, seed=32, device=gpu)
    toks = [int(t) for t in np.random.default_rng(6).integers(0, spec.vocab_size, 2100)]
    a, b = _both(monkeypatch, img, spec, lambda m: m.prefill_gemm(toks, 0), len(toks))
    for l, (x, y) in enumerate(zip(a, b)):
        np.testing.assert_allclose(x, y, rtol=0, atol=2 * KV_ATOL_GEMM * (4 if spec.quant else 1), err_msg=f"layer {l}")


@pytest.mark.parametrize("name", ["gqa-half", "mha-interleaved"])
def test_scales_follow_weights_and_cache(gpu, name, monkeypatch):
    """Weight rows between 2^-20 and 2^20 of their usual size (scales of the rows and of the gated unit), a zero row, and
    cache rows of 1e6 in front of the prompt (scales of the attention output).  Rows are held to 2e-5 of their largest entry:
    2^-24 per operand, 2^-22 per product, some hundred roundings to fp32 behind them.  What lies far below the largest entry
    is held by test_pair_exact_gpu.py."""
    spec = dataclasses.replace(SPECS[name], seq_len=512)
    img = binfmt.synth_image(spec, seed=33, device=gpu)
    for e in binfmt.layout(spec)[0]:
        base = e.name.split(".")[0]
        if base in ("wo", "w2", "w3"):
            w = binfmt.tensor_from_image(img, e)
            k = torch.arange(e.shape[0], device=gpu) % 41 - 20
            w.copy_(w * torch.exp2(k.float())[:, None] * 2.0 ** -20)
            w[1].zero_()
    rng = np.random.default_rng(7)
    toks = [int(t) for t in rng.integers(0, spec.vocab_size, 150)]
    old = 40
    k0 = rng.standard_normal((old, spec.kv_dim)).astype(np.float32)
    v0 = (1e6 * rng.standard_normal((old, spec.kv_dim))).astype(np.float32)

    def run(m):
        for l in range(spec.n_layers):
            m.write_kv(l, 0, k0, v0)
        m.prefill_gemm(toks, old)

    a, b = _both(monkeypatch, img, spec, run, old + len(toks))
    for l, (x, y) in enumerate(zip(a, b)):
        assert np.isfinite(x).all()
        top = np.abs(y).max(axis=1, keepdims=True)
        assert (np.abs(x - y) / top).max() < 2e-5, (l, float((np.abs(x - y) / top).max()))
