"""Per-token kernels of layer-list prompts (csrc/kh_lops.h, kh_latent.h, kh_scan.h) and the attention of four sets of waves
(csrc/kh_heads.h): rows with and without a remainder, segments shorter than the convolution, launches that leave CUs idle."""
import pytest

import layers_util as U
from kuiperllama_amd import _ffi

pytestmark = pytest.mark.gpu
BOTH = pytest.mark.parametrize("dtype", ["float32", "bfloat16"])


def _prompt(mod, dtype, n, cuts, **kw):
    m = mod.load(dtype, **kw)
    toks = mod.tokens(n)
    U.check(U.run_alone(m, toks, cuts), mod.logits(toks), dtype, f"{n} {cuts}")
    m.close()


@BOTH
@pytest.mark.parametrize("q_rank,kv_rank,rot", [(1024, 512, 64), (2044, 40, 12), (2052, 36, 6), (2300, 260, 10), (1026, 64, 8)])
def test_latent_rows(gpu, dtype, q_rank, kv_rank, rot):
    """In registers, beyond them, quads that the rotated part does not fill, and rows that are no quads."""
    _prompt(U.Model(U.config([U.latent(2, 20, rot, 28, kv_rank, q_rank, 0.3)], width=48, vocab=60)), dtype, 40, (7, 8, 30))


@BOTH
@pytest.mark.parametrize("inner,conv", [(72, 4), (75, 4), (2060, 4), (72, 2), (40, 6)])
def test_convolution_state(gpu, dtype, inner, conv):
    """Pieces of one, two and three tokens behind one another, where the state is made of the state before it."""
    _prompt(U.Model(U.config([U.mamba(inner, 5, 3, conv), U.mamba(24, 3, 2, 4)], width=40, vocab=50)), dtype, 150, (1, 2, 4, 7, 70, 135))


@BOTH
@pytest.mark.parametrize("top", [4, 5, 8, 9])
def test_rows_of_experts(gpu, dtype, top):
    """Chosen rows in batches of four, with outputs that are no stored row among them."""
    _prompt(U.Model(U.config([U.with_ff(U.mamba(), experts=9, identity=3, top=top, ff=20)], width=1100, vocab=60)), dtype, 33, (20,))


@BOTH
@pytest.mark.parametrize("experts,top,n", [(4, 2, 240), (3, 1, 345), (5, 1, 610), (2, 1, 490)])
def test_expert_shares_below_an_edge(gpu, dtype, experts, top, n):
    """Shares just below 128 and 256 rows, spread by the choices: tiles of few and of many 16-row units."""
    _prompt(U.Model(U.config([U.with_ff(U.mamba(), experts=experts, top=top, ff=72)], width=136, vocab=60)), dtype, n, (), max_seq_len=640)


@BOTH
@pytest.mark.parametrize("ff,n", [(512, 1100), (512, 1036), (1024, 540)])
def test_expert_tiles_of_192_rows_in_one_round(gpu, dtype, ff, n):
    """Shares just below 256 and 128 rows whose tiles of 128 would be a second round of workgroups: the tiles that the rule of
    csrc/kh_lgemm.h::lg_group_bm makes 192 rows long, of experts with two tiles and with one, below and beyond their share."""
    width, size = 136, {"bfloat16": 2, "float32": 4}[dtype]
    assert _ffi.plan_expert_rows(7 * n, 32, 32, 2 * ff, 32 * 2 * ff * width * size) == 192
    _prompt(U.Model(U.config([U.with_ff(U.mamba(), experts=32, top=7, ff=ff)], width=width, vocab=60)), dtype, n, (), max_seq_len=1152)


@pytest.mark.parametrize("dim,vdim,window,n,cuts", [(128, 128, 40, 65, ()), (128, 128, 600, 700, (63, 64, 400)), (100, 90, 200, 300, (129,)),
                                                    (128, 128, 700, 33, (1, 2)), (65, 128, 31, 200, (31, 190))])
def test_heads_of_four_sets(gpu, dim, vdim, window, n, cuts):
    """bf16 heads of 65 to 128 columns: fewer key tiles than sets, masks inside a set's tile, rows in front of the piece."""
    layers = [U.windowed(8, 2, dim, vdim, 0.1, window, 20, 50.0), U.chunked(4, 1, dim, vdim, 0.1, window)]
    _prompt(U.Model(U.gusorax(layers, width=64, vocab=70, positions=800)), "bfloat16", n, cuts, max_seq_len=800)


@pytest.mark.parametrize("dtype,n", [("float32", 1024), ("bfloat16", 2048)])
def test_latent_steps_of_many_splits(gpu, dtype, n):
    """Steps of one and of four sequences around 64 filled splits of one key tile, in lanes and beyond them."""
    import numpy as np
    mod = U.Model(U.config([U.latent(3, 20, 8, 28, 72, 40, 0.4)], width=40, vocab=50))
    m = mod.load(dtype, max_seq_len=n + 16)
    toks = mod.tokens(n + 3)
    want = mod.logits(toks)
    for others in (0, 3):
        s = m.open_seq()
        rest = [m.open_seq() for _ in range(others)]
        m.forward([(s, toks[:n - 2], [n - 3])])
        for i in range(n - 2, n + 3):
            got = m.forward([(s, [toks[i]], [0])] + [(r, [toks[i]], [0]) for r in rest])
            U.check(np.asarray(got)[:1], want[i:i + 1], dtype, f"{i} {others}")
        for r in [s] + rest:
            m.close_seq(r)
    m.close()


@BOTH
@pytest.mark.parametrize("inner,state", [(72, 5), (2050, 16)])
def test_scans_that_continue(gpu, dtype, inner, state):
    """Pieces of several chunks behind others, of two and of one chunk more: the same bits every time."""
    import numpy as np
    mod = U.Model(U.config([U.mamba(inner, state, 3, 4), U.mamba(24, 3, 2, 4)], width=40, vocab=50))
    toks = mod.tokens(330)
    want = mod.logits(toks)
    m = mod.load(dtype)
    out = [U.run_alone(m, toks, (70, 199, 200, 265)) for _ in range(5)]
    m.close()
    U.check(out[0], want, dtype)
    for o in out[1:]:
        np.testing.assert_array_equal(o, out[0])
