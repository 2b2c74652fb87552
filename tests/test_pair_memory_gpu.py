"""Memory of prompt passes (csrc/kh_model_prefill.hip::ensure_pg_buffers, csrc/kh_model_pair.hip::pair_prepare)."""
import numpy as np
import pytest
import torch

from kuiperllama_amd import binfmt
from test_model_gpu import KV_ATOL_GEMM

pytestmark = pytest.mark.gpu

SPEC = binfmt.ModelSpec(1024, 4096, 2, 16, 4, 500, 2304, True, binfmt.FAMILY_LLAMA, False, 64, binfmt.ROPE_HALF, 10000.0, 1e-5,
                        "pair-memory")  # 128 more slab rows are more than 6 MB


def _tokens(n):
    return [int(t) for t in np.random.default_rng(23).integers(0, SPEC.vocab_size, n)]


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_a_growing_conversation_allocates_seldom(gpu):
    from kuiperllama_amd.model import KuiperModel
    img = binfmt.synth_image(SPEC, seed=61, device=gpu)
    m = KuiperModel.from_device_image(img, SPEC)
    free = []
    for n in (400, 600, 700, 800, 900, 1000):
        m.prefill_gemm(_tokens(n), 0)
        free.append(_free())
    m.prefill_gemm(_tokens(1000), 1200)
    m.close()
    assert len(set(free[1:])) <= 2, free  # 600: 1024 rows, and K / V as pairs; once behind it twice as many of those


def test_prompt_without_memory_for_long_passes(gpu, monkeypatch):
    """1500 tokens in passes of 512 where memory for more rows is refused (KH_PG_ROWS), with the rows of one pass; and 512 slab
    rows only where no pass can be longer: the fp32-MFMA GEMMs."""
    from kuiperllama_amd.model import KuiperModel
    img = binfmt.synth_image(SPEC, seed=62, device=gpu)
    toks = _tokens(1500)
    rows, used = [], []
    for hook in (None, "KH_PG_ROWS", "KH_PG_PAIR"):
        if hook:
            monkeypatch.setenv(hook, "512" if hook == "KH_PG_ROWS" else "0")
        m = KuiperModel.from_device_image(img, SPEC)
        m.prefill_gemm(toks[:20], 0)
        before = _free()
        m.prefill_gemm(toks, 0)
        used.append(before - _free())
        rows.append(m.read_kv(1, 0, 1500))
        m.close()
        if hook:
            monkeypatch.delenv(hook)
    for other in rows[1:]:
        for a, b in zip(rows[0], other):
            np.testing.assert_allclose(a, b, rtol=0, atol=2 * KV_ATOL_GEMM)
    slabs = 1536 * (4 * SPEC.dim + SPEC.hidden_dim) * 4
    assert used[0] >= slabs and used[1] < slabs and used[2] < slabs, used
