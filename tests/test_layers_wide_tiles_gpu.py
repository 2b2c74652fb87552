"""Plain bf16 GEMMs of prompts in workgroups of eight waves (csrc/kh_lgemm.h): where the tiles fill the CUs once, as 128 x 128 or
256 x 256, at both ends of their ranges, with fewer stages of K than the ring has and with more, ragged tokens and features."""
import pytest

import layers_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,inner,n", [(40, 2700, 257), (700, 2700, 300), (90, 5500, 384), (300, 8190, 255),  # 129 ... 256 tiles
                                           (700, 2690, 250), (40, 5500, 385),                                  # one tile outside
                                           (64, 8576, 700), (330, 10900, 767), (50, 8576, 613)])               # 201, 256, too empty
def test_prompts(gpu, width, inner, n):
    mod = U.Model(U.config([U.mamba(inner=inner, state=1, dt_rank=1, conv=1), U.mamba(inner=20)], width=width, vocab=37))
    toks = mod.tokens(n)
    m = mod.load("bfloat16", max_seq_len=800)
    U.check(U.run_alone(m, toks, (n - 1,))[-40:], mod.logits(toks)[-40:], "bfloat16", f"{width} {inner} {n}")
    m.close()
