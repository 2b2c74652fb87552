"""Output launch of the layer-list decode step (csrc/kh_ldecode.h, k_ld_out) at rows of several blocks and their edges (a
block is 64 x 16 bytes: 256 fp32, 512 bf16 elements): fused steps of one to four sequences against the pass kernels, which
the oracle tests hold.  fp32 storage: both accumulate in fp32, the sums differ by their order."""
import numpy as np
import pytest

from kuiperllama_amd import checkpoint
from layers_util import clamped, config, dense, gusorax, mamba, chunked, with_ff

pytestmark = pytest.mark.gpu

CASES = {
    # width 1100: padded rows of 1152, no multiple of a block
    "ff-below-block": config([with_ff(mamba(inner=520), ff=250, shared=1030, top=3)], width=1100),
    "ff-one-block": config([with_ff(mamba(inner=256), ff=256, shared=512, top=1)], width=256),
    "ff-above-block": config([with_ff(mamba(inner=1100), ff=260, shared=0, top=4)], width=514),
    "no-ff": config([mamba(inner=700)], width=130),
    "heads-dense": gusorax([dict(chunked(heads=8, dim=64, vdim=80), mlp=dense(1300)),
                            dict(chunked(heads=8, dim=64, vdim=80), mlp=clamped(7, 5, 300))], width=640),
}


@pytest.mark.parametrize("dtype,tol", [("float32", 2e-5), ("bfloat16", 3e-2)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_fused_step_against_pass(gpu, name, dtype, tol, monkeypatch):
    from kuiperllama_amd.model import KuiperModel
    cfg = CASES[name]
    img = checkpoint.safetensors_image(checkpoint.random_tensors(cfg, 3))
    rng = np.random.default_rng(4)
    for n in (1, 2, 3, 4):
        toks = rng.integers(0, cfg["vocab"], (n, 9))
        out = []
        for decode in (None, "0"):
            if decode:
                monkeypatch.setenv("KH_HY_DECODE", decode)
            m = KuiperModel.from_tensors(cfg, img, max_seq_len=64, dtype=dtype, max_seqs=n)
            from kuiperllama_amd import _ffi
            _ffi.sync_env()
            seqs = [m.open_seq() for _ in range(n)]
            m.forward([(s, t[:5], []) for s, t in zip(seqs, toks)])
            out.append(np.stack([m.forward([(s, [t[i]], [0]) for s, t in zip(seqs, toks)]) for i in range(5, 9)]))
            m.close()
            monkeypatch.delenv("KH_HY_DECODE", raising=False)
        _ffi.sync_env()
        a, b = out
        assert np.abs(a - b).max() <= tol * max(1.0, np.abs(b).max()), (n, float(np.abs(a - b).max()), float(np.abs(b).max()))
