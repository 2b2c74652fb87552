"""Host-side launch planning (no GPU): the decode GEMV shapes (csrc/kh_model_step.hip::pick_shape) and the
prefill GEMM shapes (csrc/kh_model_prefill.hip::pg_shape) through the host-only C-ABI entries
kh_plan_decode_shapes / kh_plan_pair_shapes / kh_plan_prefill_shape.  Invariants every plan must satisfy for every BASELINE
geometry, plus the plans DESIGN.md documents (so that a change of the heuristics shows up here and not
only as a slower GPU run)."""
import itertools

import pytest

from kuiperllama_amd import _ffi, binfmt

PRESETS = ["llama3.2-1b", "llama2-7b", "llama2-7b-int8", "qwen2.5-0.5b", "tinyllama-1.1b"]


@pytest.mark.parametrize("name", PRESETS)
def test_decode_plan_invariants(name):
    sp = binfmt.PRESETS[name]
    plan = _ffi.plan_decode_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.vocab_size, sp.quant)
    rows = {"qkv": sp.dim + 2 * sp.kv_dim, "wo": sp.dim, "ffn13": 2 * sp.hidden_dim, "w2": sp.dim,
            "cls": sp.vocab_size}
    cols = {"qkv": sp.dim, "wo": sp.dim, "ffn13": sp.dim, "w2": sp.hidden_dim, "cls": sp.dim}
    max_split = {"qkv": 2, "wo": 4, "ffn13": 1, "w2": 4, "cls": 1}
    for k, s in plan.items():
        assert s["split"] in (1, 2, 4) and s["split"] <= max_split[k], (k, s)
        # int8 w2 alone may take two exact tiles of three loads per row (round 6, profiles/r6_w2_u3_ab.txt)
        assert s["u"] in (((2, 3, 4) if k == "w2" else (2, 4)) if sp.quant else (2, 4, 8)), (k, s)
        assert s["wg"] in (256, 512), (k, s)
        assert 1 <= s["grid"] <= 1024, (k, s)  # never more than 4 x 256-thread workgroups per CU
        # a split part still streams a useful number of bytes per row pair
        elem = 1 if sp.quant else 4
        assert s["split"] == 1 or 2 * cols[k] * elem // s["split"] >= (4096 if sp.quant else 8192), (k, s)
        # the grid never exceeds the work: one workgroup handles >= one row pair per wave group
        pairs_per_wg = (s["wg"] // 64) // s["split"]
        pairs = (rows[k] // 2 + 1) // 2 if k == "ffn13" else (rows[k] + 1) // 2
        assert s["grid"] <= -(-max(pairs, 1) // pairs_per_wg) or s["grid"] % 256 == 0, (k, s)


@pytest.mark.parametrize("arch,width,elem,tokens,rows", [
    # a second round of 128-row tiles, one round of 192-row tiles
    ("gusorax", 1024, 2, 1036, 192), ("gusorax", 1024, 2, 1100, 192), ("gusorax", 1024, 4, 1100, 192), ("gusorax", 1024, 2, 1165, 192),
    ("gufanex", 1024, 2, 1360, 192), ("gufanex", 1024, 4, 1450, 192),
    # one round of either
    ("gusorax", 512, 2, 540, 128), ("gusorax", 512, 4, 1100, 128), ("gusorax", 512, 4, 1700, 128), ("gusorax", 1024, 4, 540, 128),
    ("gufanex", 512, 2, 700, 128), ("gufanex", 512, 2, 1450, 128), ("gufanex", 1024, 4, 700, 128),
    # shares far below the edge, more than one round of 192, more weights than two stages cover
    ("gusorax", 1024, 2, 800, 128), ("gusorax", 1024, 2, 1000, 128), ("gusorax", 1024, 2, 1700, 128), ("gusorax", 2048, 2, 1100, 128),
    ("gufanex", 2048, 2, 740, 128), ("gusorax", 1024, 2, 290, 64), ("gusorax", 1024, 2, 100, 32)])
def test_expert_tiles_take_192_rows_for_a_second_round_alone(arch, width, elem, tokens, rows):
    """32 experts of half a width, 7 of 32 outputs chosen (Gusorax) or 6 of 36 (Gufanex)."""
    top, outputs = (7, 32) if arch == "gusorax" else (6, 36)
    assert _ffi.plan_expert_rows(tokens * top, outputs, 32, width, 32 * width * width * elem) == rows


@pytest.mark.parametrize("width,ff,f32,tokens,beside", [
    (1024, 256, False, 1100, False), (2048, 256, False, 400, False), (2048, 256, True, 17, False), (2048, 256, True, 100, False),
    (2048, 256, True, 400, True), (2048, 4096, False, 17, True), (2048, 4096, False, 400, True), (1024, 3584, False, 17, False),
    (1024, 3584, False, 1100, True)])
def test_mixers_run_beside_a_dense_feed_forward_of_some_size(width, ff, f32, tokens, beside):
    """Heads of 128, a quarter of them with keys and values.  The shorter branch pays for the events: a short feed-forward gains
    nothing beside a mixer however long that is."""
    mixer = width * (2 * width + 2 * width // 4 + width)
    assert _ffi.plan_mixer_beside(mixer, 3 * width * ff, 0, 0, 0, 0, tokens, f32) is beside
    assert not _ffi.plan_mixer_beside(100 * mixer, 3 * 64 * 256, 0, 0, 0, 0, tokens, f32)


def test_mixers_run_beside_experts():
    """Experts are launches enough for a mixer of any size: what counts is the layer's work in all."""
    gusorax = lambda width, tokens, mixer=None: _ffi.plan_mixer_beside(  # noqa: E731
        3 * width * width if mixer is None else mixer, 0, 3 * width * width // 2, 32, 7, 32, tokens, False)
    assert [gusorax(1024, t) for t in (1, 3, 17, 150, 1100)] == [False, False, True, True, True]
    assert [gusorax(1024, t, 4 * 64 * 1024) for t in (17, 1100)] == [True, True]
    assert not gusorax(512, 50) and gusorax(512, 1100)


@pytest.mark.parametrize("vocab", [32000, 151936])
@pytest.mark.parametrize("dim,grid", [(192, 512), (288, 512), (336, 512), (384, 256), (448, 256), (512, 256), (896, 256)])
def test_classifiers_of_short_rows(dim, grid, vocab):
    """fp32 rows of less than 1.5 KB: 16 waves a CU, in workgroups of 512 threads like the longer ones."""
    cls = _ffi.plan_decode_shapes(dim, 3 * dim, dim, vocab, False)["cls"]
    assert (cls["grid"], cls["wg"], cls["split"]) == (grid, 512, 1)


@pytest.mark.parametrize("name,narrow,wide", [("tinyllama-1.1b", (17, 32), (33, 50, 64)), ("qwen2.5-0.5b", (17, 32), (33, 41, 64))])
def test_gated_tiles_of_short_prompts(name, narrow, wide):
    """w1 + w3: tiles of 64 rows only where they win by more than their finer scales cost the product behind them."""
    sp = binfmt.PRESETS[name]
    bn = lambda n: _ffi.plan_pair_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, False, n)["w13"]["bn"]  # noqa: E731
    assert [bn(n) for n in narrow] == [64] * len(narrow) and [bn(n) for n in wide] == [128] * len(wide)


@pytest.mark.parametrize("head_size", [48, 64])
def test_attention_and_wo_in_one_round_of_workgroups(head_size, monkeypatch):
    """A CU holds one of its workgroups: never more than 256, every row somebody's; and what does not take the joint launch."""
    monkeypatch.delenv("KH_ATTN_WO", raising=False)
    taken = 0
    for heads in range(1, 45):
        for kv in range(1, heads + 1):
            if heads % kv:
                continue
            dim = heads * head_size
            p = _ffi.plan_attn_wo(dim, 11 * dim // 4 // 16 * 16 + 16, heads, kv, 512)
            if kv > 8 or heads // kv * head_size > 512 or dim > 2048:
                assert p == dict(end=0, parts=0, rows=0, workgroups=0), (heads, kv, p)
            elif p["end"]:
                taken += 1
                assert p["parts"] == kv and p["end"] <= 256
                assert p["workgroups"] == kv * -(-dim // p["rows"]) <= 256, (heads, kv, p)
    assert taken > 40
    assert not _ffi.plan_attn_wo(2048, 8192, 32, 8, 512, True)["end"] and not _ffi.plan_attn_wo(2048, 8192, 16, 8, 512)["end"]


def test_attention_and_wo_in_one_launch_as_far_as_it_pays(monkeypatch):
    """The presets take it at all positions below 256; geometries of many parts as far as they gain."""
    monkeypatch.delenv("KH_ATTN_WO", raising=False)
    for name, end in (("stories15M", 256), ("qwen2.5-0.5b", 256), ("tinyllama-1.1b", 256), ("llama3.2-1b", 256), ("llama2-7b", 0)):
        sp = binfmt.PRESETS[name]
        assert _ffi.plan_attn_wo(sp.dim, sp.hidden_dim, sp.n_heads, sp.n_kv_heads, 512)["end"] == end, name
    for size, heads, kv, end in ((64, 8, 1, 256), (64, 14, 2, 256), (64, 18, 3, 256), (64, 15, 5, 128), (64, 20, 5, 128), (64, 8, 4, 256), (64, 16, 4, 192),
                                 (64, 12, 6, 192), (64, 18, 6, 64), (64, 14, 7, 128), (64, 21, 7, 64), (64, 8, 8, 256), (64, 16, 8, 128), (64, 24, 8, 256),
                                 (48, 30, 5, 256), (48, 18, 6, 256), (48, 24, 6, 128), (48, 21, 7, 256), (48, 28, 7, 64), (48, 16, 8, 256), (48, 24, 8, 0)):
        assert _ffi.plan_attn_wo(size * heads, 8192, heads, kv, 512)["end"] == end, (size, heads, kv)
    for dim, hidden, heads, kv, end in ((1536, 4096, 24, 8, 64), (1536, 3072, 24, 8, 128), (1536, 4096, 24, 4, 256), (2048, 4096, 32, 8, 64),
                                        (2048, 4096, 32, 4, 256), (1536, 4224, 24, 8, 256)):  # 1024, 768 or 512 workgroups in ffn13
        assert _ffi.plan_attn_wo(dim, hidden, heads, kv, 512)["end"] == end, (dim, hidden, kv)
    assert _ffi.plan_attn_wo(2048, 8192, 32, 8, 512)["end"] == 256 and _ffi.plan_attn_wo(2048, 8192, 32, 8, 100)["end"] == 256
    monkeypatch.setenv("KH_ATTN_WO", "100")
    assert _ffi.plan_attn_wo(64 * 16, 2816, 16, 8, 512)["end"] == 100
    monkeypatch.setenv("KH_ATTN_WO", "0")
    assert _ffi.plan_attn_wo(2048, 8192, 32, 8, 512)["end"] == 0


def test_decode_plan_int8_wide_rows_keep_the_small_tile():
    """int8 rows that need more than four 16-byte loads per lane walk several tiles of TWO loads (qkv / wo / ffn13 /
    cls; w2 takes two tiles of three where that is exact) - never the fp32 rule's 4 or 8.  Geometries wider than any
    preset, so that the branch is exercised (a dangling `else` once sent every int8 launch but w2 through the fp32
    rule: invisible at the presets, whose int8 rows need at most four loads per lane)."""
    for dim, hidden in ((8192, 28672), (6144, 16384), (5120, 13824)):
        plan = _ffi.plan_decode_shapes(dim, hidden, dim, 32000, True)
        for k, s in plan.items():
            per_lane = -(-(-(-(hidden if k == "w2" else dim) // 16 // s["split"])) // 64)
            if per_lane > 4:
                want = (3,) if k == "w2" and per_lane <= 6 else (2,)
                assert s["u"] in want, (dim, hidden, k, s, per_lane)
            assert s["u"] in (2, 3, 4), (k, s)
    # fp32 keeps its own rule: eight loads per lane when the row covers them
    assert _ffi.plan_decode_shapes(8192, 28672, 8192, 32000, False)["ffn13"]["u"] == 8


def test_decode_plan_documented_shapes(monkeypatch):
    """The shapes DESIGN.md 3.2 quotes for the two bench workloads."""
    for k in ("QKV", "WO", "FFN", "W2", "CLS"):
        monkeypatch.delenv("KH_SHAPE_" + k, raising=False)
    sp = binfmt.PRESETS["llama2-7b-int8"]
    plan = _ffi.plan_decode_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.vocab_size, True)
    assert plan["qkv"] == {"split": 1, "u": 4, "grid": 512, "wg": 256}
    assert plan["wo"] == {"split": 1, "u": 4, "grid": 512, "wg": 256}
    assert plan["ffn13"] == {"split": 1, "u": 4, "grid": 512, "wg": 256}
    assert plan["w2"] == {"split": 2, "u": 3, "grid": 512, "wg": 512}  # 5.4 loads per lane: two tiles of three
    assert plan["cls"] == {"split": 1, "u": 4, "grid": 512, "wg": 256}
    sp = binfmt.PRESETS["llama3.2-1b"]
    plan = _ffi.plan_decode_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.vocab_size, False)
    assert plan["ffn13"] == {"split": 1, "u": 8, "grid": 512, "wg": 256}  # the roofline kernel of bench.py
    assert plan["w2"]["wg"] == 512 and plan["cls"]["wg"] == 512
    # the tuning hook is honoured, and a malformed value is ignored
    monkeypatch.setenv("KH_SHAPE_FFN", "1,4,256")
    assert _ffi.plan_decode_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.vocab_size, False)["ffn13"] == \
        {"split": 1, "u": 4, "grid": 256, "wg": 256}
    monkeypatch.setenv("KH_SHAPE_FFN", "3,4,256")
    assert _ffi.plan_decode_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.vocab_size, False)["ffn13"] == plan["ffn13"]


@pytest.mark.parametrize("name", PRESETS)
def test_prefill_plan_invariants(name):
    sp = binfmt.PRESETS[name]
    kq = 64 if sp.quant else 16
    gemms = [("qkv", sp.dim + 2 * sp.kv_dim, sp.dim, sp.dim % 32 == 0 and sp.kv_dim % 32 == 0),
             ("resid", sp.dim, sp.dim, sp.dim % 32 == 0), ("resid", sp.dim, sp.hidden_dim, sp.dim % 32 == 0),
             ("swiglu", sp.hidden_dim, sp.dim, sp.hidden_dim % 32 == 0)]
    for (epi, rows, K, r2), T in itertools.product(gemms, (1, 16, 17, 64, 100, 128, 129, 256, 300, 384, 512)):
        p = _ffi.plan_prefill_shape(epi, T, rows, K, sp.quant, r2)
        nm = 2 if epi == "swiglu" else 1
        assert (p["R"], p["NT"]) in ((2, 8), (2, 4), (2, 2), (1, 4)), (epi, T, p)
        assert p["R"] == 1 or r2
        assert p["slices"] * p["NT"] * 16 >= T and (p["slices"] - 1) * p["NT"] * 16 < T, (epi, T, p)
        assert p["slices"] * p["NT"] * 16 <= -(-T // 128) * 128  # inside the slab stride of the pass
        assert p["ks"] in (1, 2, 4, 8) and p["ks"] * nm * 64 <= 512, (epi, T, p)
        assert p["kz"] in (1, 2, 4) and (p["kz"] == 1 or epi == "resid"), (epi, T, p)
        # every wave keeps a useful K range (fp32: 16 blocks of 16 columns; int8: 4 blocks of 64)
        assert p["ks"] * p["kz"] == 1 or (K // kq) // (p["ks"] * p["kz"]) >= (4 if sp.quant else 16), (epi, T, p)
        assert p["workgroups"] == rows // (16 * p["R"]) * p["slices"] * p["kz"]
        # one workgroup per CU at a time: fp32 launches of more than 256 workgroups only
        assert not p["solo"] or (not sp.quant and p["workgroups"] > 256), (epi, T, p)


def test_prefill_plan_documented_shapes(monkeypatch):
    """Llama-3.2-1B, DESIGN.md 3.5: a 512-token pass puts every GEMM on the big tile; a 128-token pass splits
    the K range of wo / w2 across two workgroups; KH_PG_KZ=0 / KH_PG_SOLO=0 are read at load time and are not
    exercised here."""
    sp = binfmt.PRESETS["llama3.2-1b"]
    f = lambda epi, T, rows, K: _ffi.plan_prefill_shape(epi, T, rows, K, False, True)  # noqa: E731
    assert f("swiglu", 128, sp.hidden_dim, sp.dim) == dict(R=2, NT=8, ks=2, slices=1, solo=0, kz=1, workgroups=256)
    assert f("swiglu", 512, sp.hidden_dim, sp.dim) == dict(R=2, NT=8, ks=2, slices=4, solo=1, kz=1, workgroups=1024)
    for K in (sp.dim, sp.hidden_dim):
        assert f("resid", 512, sp.dim, K) == dict(R=2, NT=8, ks=4, slices=4, solo=0, kz=1, workgroups=256)
        p = f("resid", 128, sp.dim, K)
        assert p["kz"] == 2 and p["workgroups"] == 256 and p["solo"] == 0
    assert f("qkv", 512, sp.dim + 2 * sp.kv_dim, sp.dim)["solo"] == 1
    # Llama-2-7B fp32, 128 tokens: four-wave workgroups, one per CU at a time (was 344 two-wave workgroups)
    s7 = binfmt.PRESETS["llama2-7b"]
    p = f("swiglu", 128, s7.hidden_dim, s7.dim)
    assert (p["R"], p["NT"], p["ks"], p["solo"]) == (2, 8, 2, 1)
    # argument errors
    with pytest.raises(_ffi.KhError):
        _ffi.plan_prefill_shape("qkv", 513, 3072, 2048, False, True)
    with pytest.raises(_ffi.KhError):
        _ffi.plan_prefill_shape("qkv", 128, 3072, 2040, False, True)


@pytest.mark.parametrize("name", PRESETS + ["stories15M"])
def test_pair_plan_invariants(name):
    """The GEMMs that prompts run on (csrc/kh_model_pair.hip): tiles that exist, K slices of four stages at least and of the
    residual products only, no fewer workgroups at more tokens with the same tile."""
    sp = binfmt.PRESETS[name]
    tiles = ((112, 128), (64, 128), (32, 128), (128, 256)) if sp.quant else ((128, 128), (64, 128), (32, 128), (32, 64))
    N = {"qkv": sp.dim + 2 * sp.kv_dim, "wo": sp.dim, "w13": 2 * sp.hidden_dim, "w2": sp.dim}
    last = {}
    for T in (1, 16, 17, 32, 33, 64, 65, 112, 113, 128, 200, 256, 300, 511, 512, 777, 1024, 1900, 2048):
        for g, p in _ffi.plan_pair_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, sp.quant, T).items():
            K = sp.hidden_dim if g == "w2" else sp.dim
            assert (p["bm"], p["bn"]) in tiles, (T, g, p)
            assert p["kz"] in ((1, 2, 4) if g in ("wo", "w2") else (1,)), (T, g, p)
            assert p["kz"] == 1 or K // (64 if sp.quant else 32) // p["kz"] >= 4, (T, g, p)
            assert p["workgroups"] == -(-N[g] // p["bn"]) * -(-T // p["bm"]) * p["kz"], (T, g, p)
            shape = (p["bm"], p["bn"], p["kz"])
            assert last.get((g, shape), 0) <= p["workgroups"], (T, g, p)
            last[g, shape] = p["workgroups"]


def test_pair_plan_of_prompts(monkeypatch):
    """Llama-3.2-1B and Llama-2-7B int8: the plans that the measured prompt times belong to."""
    sp = binfmt.PRESETS["llama3.2-1b"]
    p = _ffi.plan_pair_shapes(sp.dim, sp.hidden_dim, sp.kv_dim, False, 512)
    assert p == {"qkv": dict(bm=64, bn=128, kz=1, workgroups=192), "wo": dict(bm=64, bn=128, kz=2, workgroups=256),
                 "w13": dict(bm=128, bn=128, kz=1, workgroups=512), "w2": dict(bm=64, bn=128, kz=4, workgroups=512)}
    s7 = binfmt.PRESETS["llama2-7b-int8"]
    p = _ffi.plan_pair_shapes(s7.dim, s7.hidden_dim, s7.kv_dim, True, 777)
    assert _ffi.plan_pair_shapes(16384, 53248, 1024, False, 512) and _ffi.plan_pair_shapes(18432, 73728, 2304, True, 512)
    assert p["w13"] == dict(bm=112, bn=128, kz=1, workgroups=1204) and p["qkv"]["workgroups"] == 672
    for bad in ((2048, 8192, 512, False, 0), (2048, 8192, 512, False, 2049), (2064, 8192, 512, False, 512), (2080, 8192, 512, True, 512),
                (18432, 73728, 2304, False, 512), (18432, 245760, 2304, True, 512)):  # matrices of more than 4 GiB
        with pytest.raises(_ffi.KhError):
            _ffi.plan_pair_shapes(*bad)


def test_attention_plan_and_split_geometry(monkeypatch):
    """The decode-attention geometry (kh_attn.h::attn_plan / attn_split_len / attn_active_splits - host AND device
    code) through the host-only kh_plan_attention: the Llama-3.2-1B, Qwen2.5-0.5B, Llama-2-7B and tiny-head plans, the
    per-head / group switch, and the split arithmetic at EVERY position of a long cache against its definition
    (split length = ceil(timesteps / splits) rounded up to 64, at least 256; active = ceil(timesteps / length)) -
    the device takes a division-free shortcut for timesteps <= 256 * splits that must give the same values."""
    from kuiperllama_amd import _ffi
    monkeypatch.delenv("KH_ATTN_TLONG", raising=False)
    a = _ffi.plan_attention(32, 4, 64, 131072, 63)          # Llama-3.2-1B
    assert (a["ns"], a["ns_g"], a["stride"], a["t_long"]) == (16, 32, 32, 4096)
    assert (a["group_path"], a["active_splits"], a["split_len"], a["workgroups"]) == (0, 1, 256, 32)
    assert _ffi.plan_attention(32, 4, 64, 131072, 4094)["workgroups"] == 32 * 16
    b = _ffi.plan_attention(32, 4, 64, 131072, 4095)        # first position of the group path
    assert (b["group_path"], b["active_splits"], b["workgroups"]) == (1, 16, 8 * 16)
    assert _ffi.plan_attention(32, 4, 64, 131072, 131071)["workgroups"] == 8 * 32
    q = _ffi.plan_attention(14, 7, 64, 32768, 32767)        # Qwen2.5-0.5B: 2 KV heads cannot fill the chip with groups
    assert q["ns_g"] == 0 and q["group_path"] == 0 and q["active_splits"] == 16 and q["split_len"] == 2048
    assert _ffi.plan_attention(32, 1, 128, 4096, 4095)["ns_g"] == 0   # MHA: no group path
    assert _ffi.plan_attention(6, 1, 32, 256, 255)["ns"] == 1          # head size <= 32: generic kernel, no splits
    monkeypatch.setenv("KH_ATTN_TLONG", "300")               # the hook moves the switch point
    assert _ffi.plan_attention(32, 4, 64, 3000, 299)["group_path"] == 1
    assert _ffi.plan_attention(32, 4, 64, 3000, 298)["group_path"] == 0
    monkeypatch.delenv("KH_ATTN_TLONG")
    for seq, heads, kvm in ((9000, 8, 1), (131072, 32, 4)):
        ns = _ffi.plan_attention(heads, kvm, 64, seq, 0)["ns"]
        step = 1 if seq < 20000 else 37
        for pos in list(range(0, seq, step)) + [seq - 1]:
            p = _ffi.plan_attention(heads, kvm, 64, seq, pos)
            n = p["ns_g"] if p["group_path"] else ns
            nt = pos + 1
            want_len = max(256, (-(-nt // n) + 63) // 64 * 64)
            assert p["split_len"] == want_len and p["active_splits"] == -(-nt // want_len), (seq, pos, p)
            assert p["active_splits"] <= n
    # head size 128 (Llama-2-7B): one split up to 256 timesteps, then a 128-timestep quantum (a split then streams the
    # 128 KiB that 256 timesteps of a 64-wide head are); KH_ATTN_TS overrides the quantum
    assert _ffi.plan_attention(32, 1, 128, 2048, 0)["ns"] == 16
    for pos, (n_want, len_want) in {63: (1, 256), 255: (1, 256), 256: (3, 128), 383: (3, 128), 384: (4, 128),
                                    1023: (8, 128), 2047: (16, 128)}.items():
        p = _ffi.plan_attention(32, 1, 128, 2048, pos)
        assert (p["active_splits"], p["split_len"], p["workgroups"]) == (n_want, len_want, 32 * n_want), (pos, p)
    ns = _ffi.plan_attention(32, 1, 128, 9000, 0)["ns"]
    for pos in range(0, 9000):
        p = _ffi.plan_attention(32, 1, 128, 9000, pos)
        nt = pos + 1
        want_len = 256 if nt <= 256 else max(128, (-(-nt // ns) + 63) // 64 * 64)
        assert p["split_len"] == want_len and p["active_splits"] == -(-nt // want_len) <= ns, (pos, p)
    monkeypatch.setenv("KH_ATTN_TS", "256")
    assert _ffi.plan_attention(32, 1, 128, 2048, 383)["active_splits"] == 2
    monkeypatch.setenv("KH_ATTN_TS", "64")
    assert _ffi.plan_attention(32, 4, 64, 131072, 383)["active_splits"] == 6
    assert _ffi.plan_attention(32, 4, 64, 131072, 255)["active_splits"] == 1
    monkeypatch.delenv("KH_ATTN_TS")


@pytest.mark.parametrize("sets", [1, 2, 4])
def test_attention_over_heads_fits_a_cu(sets):
    """Stages of every key and value size beside every distance table within the 160 KB of a CU (three stages of four sets of
    waves once left 16 KB for a table of up to 32)."""
    for key, value in itertools.product((1, 64, 65, 128, 192, 256), repeat=2):
        pad = -(-key // 64) * 64 + -(-value // 64) * 64
        if sets > 1 and pad > 256:
            with pytest.raises(_ffi.KhError):
                _ffi.plan_heads_lds(key, value, sets, 0)
            continue
        for table in (0, 4, 16384, 16388, 20000, 32764, 32768, 32772, 1 << 20):
            lds = _ffi.plan_heads_lds(key, value, sets, table)
            assert lds <= 160 * 1024, (key, value, sets, table, lds)
            stages, rest = divmod(lds - (table if table <= 32768 else 0), sets * 64 * pad)
            assert rest == 0 and stages in (2, 3)


@pytest.mark.parametrize("quant,step,most,forms", [(False, 4, 16380, 16), (True, 16, 16352, 12)])
def test_every_matmul_has_its_kernel(quant, step, most, forms):
    """kh_matmul_f32 / kh_matmul_q8: every length of the vector path and every split has a compiled kernel, and no more are
    compiled than some length reaches.  Rows around the numbers where the split changes: 2048 and 4096 waves have work."""
    seen = set()
    for M in range(step, most + 1, step):
        for K in (1, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 1 << 20):
            p = _ffi.plan_matmul(quant, M, K)
            assert p["wg"] // 64 % p["split"] == 0 and p["grid"] * (p["wg"] // 64) <= 4096 * p["split"], (M, K, p)
            assert p["staged"] == 0 or 4 * p["staged"] * p["wg"] >= M, (M, K, p)
            seen.add((p["u"], p["staged"], p["split"]))
    assert len(seen) == forms
    with pytest.raises(_ffi.KhError):
        _ffi.plan_matmul(quant, most + step, 1)
