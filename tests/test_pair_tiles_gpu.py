"""The row tiles of a prompt GEMM over the eight XCDs (csrc/kh_pair.h): fewer of them than XCDs, no multiple of eight, and token tiles of
which an XCD takes a part."""
import pytest

from kuiperllama_amd import binfmt
from test_pair_exact_gpu import errors

pytestmark = pytest.mark.gpu


def _spec(dim, hidden, heads, kv, quant=False):
    return binfmt.ModelSpec(dim, hidden, 2, heads, kv, 500, 512, not quant, binfmt.FAMILY_LLAMA, quant, 64, binfmt.ROPE_HALF, 10000.0, 1e-5,
                            f"{dim}x{hidden}")


# row tiles of 128 (64) rows: wq + wk + wv 3 (6) / 9 (18) / 10 (20), w1 + w3 5 (10) / 9 (18) / 25 (50), wo and w2 2 (4) / 6 (12) / 7 (14)
@pytest.mark.parametrize("spec", [_spec(256, 320, 4, 1), _spec(768, 576, 12, 3), _spec(896, 1600, 14, 2), _spec(768, 576, 12, 3, True)],
                         ids=lambda s: f"{s.name}{'-int8' if s.quant else ''}")
@pytest.mark.parametrize("shape", ["0,1", "1,2", "2,4", "3,1"])
@pytest.mark.parametrize("n", [17, 129, 300])
def test_every_tile_is_somebodys(gpu, spec, shape, n, monkeypatch):
    """No further from 64 bits than the fp32 matrix cores, within the bound of the other prompt shapes."""
    monkeypatch.setenv("KH_PAIR_SHAPE", shape)
    pair, fp32 = errors(monkeypatch, binfmt.synth_image(spec, seed=61, device=gpu), spec, n)
    print(f"{spec.name} {shape} {n} tokens: {pair:.3g} with pairs, {fp32:.3g} without")
    assert pair <= 1.25 * fp32
