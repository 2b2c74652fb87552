"""Input and head launches of the layer-list decode step (csrc/kh_ldecode.h, k_ld_in and k_ld_head): items dealt over at most 256
workgroups of two, three segments - fewer items than workgroups, one more than they hold once, several rounds - for one, two and four
sequences, rows of one tile and of several, both storage types."""
import numpy as np
import pytest

import layers_util as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,ff,vocab", [(72, 3, 5), (72, 391, 1023), (72, 393, 1025), (600, 2100, 4099), (1100, 700, 8300),
                                            (2100, 5000, 301), (4200, 60, 517)])
def test_items_over_workgroups(gpu, dtype, width, ff, vocab):
    moe = {"kind": "moe", "expert": {"ff": 12}, "shared": {"ff": ff}, "router": {"experts": 5, "identity": 2, "top": 3}}
    mod = U.Model(U.config([dict(U.mamba(inner=200), mlp=moe), dict(U.latent(), mlp=moe)], width=width, vocab=vocab))
    toks = mod.tokens(14)
    want = mod.logits(toks)
    m = mod.load(dtype, max_seqs=4)
    for at in ([3], [1, 6], [0, 2, 5, 9]):
        seqs = [m.open_seq() for _ in at]
        for s, n in zip(seqs, at):
            if n:
                m.forward([(s, toks[:n], [])])
        for k in range(3):
            got = m.forward([(s, [toks[n + k]], [0]) for s, n in zip(seqs, at)])
            U.check(got, want[[n + k for n in at]], dtype, f"{at}, step {k}")
        for s in seqs:
            m.close_seq(s)
    m.close()
