"""The work whose speed counts: decoding, prompts and batches of the model families, and the operator interface.

Every case is one call, or one short run of calls, of the public entry points (kuiperllama_amd.model, kuiperllama_amd.ops)
on seeded random weights of a geometry that this repository already configures.  Kinds:

  "bin"        a .bin model: generate() of `steps` forward passes behind a prompt of `prompt` tokens; the tokens and the
               last logits.  Short prompts with many steps are decoding; steps == prompt is the time to the first token.
  "prompt"     a layer-list model: one prompt through forward(), the logits of its last token.
  "serve"      a layer-list model: `seqs` prompts of different lengths in one batch, then `steps` batches of one given
               token for each sequence; all their logits.
  "generate"   a layer-list model: generate() as in "bin" (fp32 storage, whose tokens two implementations agree on).
  "operators"  one decoder layer through the operator interface, as a program that keeps its own model loop calls it.
"""
import math
import struct
import zlib

import numpy as np
import torch

# ---- geometries --------------------------------------------------------------------------------------------------------
# dim, hidden, layers, heads, kv_heads, vocab, rows of the cache, tied classifier, int8, q/k/v biases, rotate halves, theta, eps
_BIN = {
    "stories15M": (288, 768, 6, 6, 6, 32000, 256, True, False, False, False, 10000.0, 1e-5),
    "qwen2.5-0.5b": (896, 4864, 24, 14, 2, 151936, 4096, True, False, True, True, 1000000.0, 1e-6),
    "tinyllama-1.1b": (2048, 5632, 22, 32, 4, 32000, 2048, False, False, False, False, 10000.0, 1e-5),
    "llama3.2-1b": (2048, 8192, 16, 32, 8, 128256, 4096, True, False, False, True, 500000.0, 1e-5),
    "llama2-7b-int8": (4096, 11008, 32, 32, 32, 32000, 2048, False, True, False, False, 10000.0, 1e-5),
}
_GROUP = 64
_VOCAB = 32000  # of the layer-list models
_POSITIONS = 4352


class _Geom:
    def __init__(self, name):
        (self.dim, self.hidden, self.layers, self.heads, self.kv_heads, self.vocab, self.rows, self.tied, self.quant,
         self.bias, self.half, self.theta, self.eps) = _BIN[name]
        self.hs = self.dim // self.heads
        self.kv = self.hs * self.kv_heads
        d, kv, h = self.dim, self.kv, self.hidden
        self.mats = {"wq": (d, d), "wk": (kv, d), "wv": (kv, d), "wo": (d, d), "w1": (h, d), "w2": (d, h), "w3": (h, d)}

    def weight_bytes(self, n):
        return n + n // _GROUP * 4 if self.quant else 4 * n


def _layers_config(case):
    """Layers of a real model's proportions: two kinds of mixers in turn, experts of half a width."""
    width, n = case["width"], case["layers"]
    if case["arch"] == "Gusorax":
        heads = width // 128
        att = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
        window, chunk = dict(att, mask={"size": 1024}, bias_max=512), dict(att, mask={"size": 2048})
        moe = {"kind": "moe", "expert": {"ff": width // 2, "limit": 7.0}, "router": {"experts": 32, "top": 7}}
        return {"architecture": "Gusorax", "vocab": _VOCAB, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
                "embedding": {"scale": float(width) ** 0.5}, "max_positions": _POSITIONS,
                "layers": [{"type": "attention_2" if i % 2 else "attention", "mixer": chunk if i % 2 else window,
                            "mlp": {"kind": "dense", "ff": 7 * width // 2} if i == 0 else moe} for i in range(n)]}
    mlp = {"kind": "moe", "expert": {"ff": width // 2}, "shared": {"ff": width},
           "router": {"experts": 32, "identity": 4, "top": 6}}
    mamba = {"type": "mamba1", "mlp": mlp, "mixer": {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}}
    latent = {"type": "latent_attention", "mlp": mlp,
              "mixer": {"heads": width // 128, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": 1536,
                        "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}}
    return {"architecture": "Gufanex", "vocab": _VOCAB, "width": width, "norm": {"eps": 1e-5}, "logit_softcap": 30.0,
            "layers": [latent if i % 2 else mamba for i in range(n)]}


# ---- the cases ---------------------------------------------------------------------------------------------------------
def listed():
    return [
        # a small story model answers a short prompt: nothing but launches and latency
        {"name": "stories15M-decode", "kind": "bin", "model": "stories15M", "prompt": 2, "steps": 64},
        # greedy decoding from an empty context, fp32 and int8 weights: the two halves of the headline metric
        {"name": "llama3.2-1b-decode", "kind": "bin", "model": "llama3.2-1b", "prompt": 2, "steps": 48},
        {"name": "llama2-7b-int8-decode", "kind": "bin", "model": "llama2-7b-int8", "prompt": 2, "steps": 32},
        # a chat turn: a question of a few dozen tokens and the start of its answer (biases, tied classifier)
        {"name": "qwen2.5-0.5b-chat", "kind": "bin", "model": "qwen2.5-0.5b", "prompt": 41, "steps": 64},
        # time to the first token: an ordinary prompt, a ragged one that fills most of the context, int8 weights
        {"name": "llama3.2-1b-prompt-512", "kind": "bin", "model": "llama3.2-1b", "prompt": 512, "steps": 512},
        {"name": "tinyllama-prompt-1900", "kind": "bin", "model": "tinyllama-1.1b", "prompt": 1900, "steps": 1900},
        {"name": "llama2-7b-int8-prompt-777", "kind": "bin", "model": "llama2-7b-int8", "prompt": 777, "steps": 777},
        # prompts of the layer-list models: scans, latent attention and experts; windows and chunks, a ragged length
        {"name": "gufanex-prompt-2048", "kind": "prompt", "arch": "Gufanex", "width": 2048, "layers": 4, "dtype": "bfloat16",
         "prompt": 2048},
        {"name": "gusorax-prompt-1100", "kind": "prompt", "arch": "Gusorax", "width": 1024, "layers": 8, "dtype": "bfloat16",
         "prompt": 1100},
        # a server's batch: four requests of different lengths, then a token for each of them per step
        {"name": "gufanex-serve-4", "kind": "serve", "arch": "Gufanex", "width": 2048, "layers": 4, "dtype": "bfloat16",
         "seqs": 4, "prompt": 300, "steps": 16},
        # one user's answer from a layer-list model held in fp32
        {"name": "gusorax-generate-fp32", "kind": "generate", "arch": "Gusorax", "width": 1024, "layers": 8, "dtype": "float32",
         "prompt": 24, "steps": 64},
        # a program with its own model loop: the operators of one decoder layer at a position in mid-context
        {"name": "operators-layer", "kind": "operators", "model": "llama3.2-1b", "position": 700},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "chat", "prompt", "layers-prompt", "serve", "generate", "operators"])
    if kind == "operators":
        return {"kind": kind, "model": rng.choice(sorted(_BIN)), "position": log(1, 250)}
    if kind in ("decode", "chat", "prompt"):
        model = rng.choice(sorted(_BIN))
        most = {"stories15M": 250, "llama2-7b-int8": 700}.get(model, 1800)
        if kind == "decode":
            p, s = rng.randint(1, 8), rng.randint(12, 60 if model != "llama2-7b-int8" else 30)
        elif kind == "chat":
            p = log(10, min(most // 2, 200))
            s = p + rng.randint(2, 24)
        else:
            p = s = log(17, most)
        return {"kind": "bin", "model": model, "prompt": p, "steps": s}
    arch, width = rng.choice(["Gufanex", "Gusorax"]), rng.choice([512, 1024, 1536, 2048])
    case = {"arch": arch, "width": width, "layers": rng.randint(2, 4 if width > 1024 else 8)}
    if kind == "layers-prompt":
        return dict(case, kind="prompt", dtype=rng.choice(["bfloat16", "bfloat16", "float32"]), prompt=log(17, 2048))
    if kind == "serve":
        return dict(case, kind="serve", dtype="bfloat16", seqs=rng.randint(1, 6), prompt=log(8, 400), steps=rng.randint(4, 16))
    p = log(2, 200)
    return dict(case, kind="generate", dtype="float32", prompt=p, steps=p + rng.randint(8, 40))


# ---- weights and inputs: each tensor from the seed and its name ---------------------------------------------------------------
def _normal(seed, name, shape, std=1.0, mean=0.0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) << 32) + zlib.crc32(name.encode()))
    w = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=g)
    return w + mean if mean else w


def _bin_weight(g, seed, name, shape):
    """fp32; the scale of the residual products is the usual one for the depth.  The last norm's weights are centred on
    zero: a tied classifier would otherwise repeat its input token for ever."""
    base = name.split(".")[0]
    if base == "final_norm":
        return _normal(seed, name, shape, 0.5)
    if base in ("att_norm", "ffn_norm"):
        return _normal(seed, name, shape, 0.05, 1.0)
    return _normal(seed, name, shape, 0.02 / math.sqrt(2 * g.layers) if base in ("wo", "w3") else 0.02)


def _quantised(w):
    rows = w.reshape(-1, _GROUP)
    scale = rows.abs().amax(1) / 127.0
    return torch.round(rows / scale[:, None]).to(torch.int8).reshape(w.shape), scale


def _layer_weight(cfg, seed, name, shape):
    """Activations of order one: linear weights N(0, 1 / fan_in), norms around one (zero where the norm adds one)."""
    last = name.rsplit(".", 1)[-1]
    adds_one = cfg["architecture"] == "Gusorax"
    if name == "embed":
        w = _normal(seed, name, shape, 1.0 / cfg.get("embedding", {}).get("scale", 1.0))
    elif adds_one and (last == "norm1" or name == "final.norm"):
        w = _normal(seed, name, shape, 0.1)
    elif name == "pos":
        w = _normal(seed, name, shape, 0.3)
    elif last == "rel":
        w = _normal(seed, name, shape)
    elif name.endswith("norm") or last in ("norm1", "norm2", "D"):
        w = _normal(seed, name, shape, 0.1, 1.0)
    elif last == "A_log":
        w = torch.log(torch.arange(1, shape[1] + 1, device="cuda").float())[None, :] + _normal(seed, name, shape, 0.1)
    elif name.endswith("dt.b"):
        w = _normal(seed, name, shape, 1.0, -3.0)
    elif last == "conv":
        w = _normal(seed, name, shape, 0.5)
    elif last == "correction":
        w = _normal(seed, name, shape, 0.02)
    elif len(shape) == 1:
        w = _normal(seed, name, shape, 0.1)
    else:
        w = _normal(seed, name, shape, shape[-1] ** -0.5)
    return w.to(torch.bfloat16)


def _tokens(seed, name, n, vocab):
    return [int(t) for t in np.random.default_rng([int(seed), zlib.crc32(name.encode())]).integers(0, vocab, n)]


def _requests(case, seed):
    """Prompts of the sequences (lengths from a quarter of `prompt` to all of it) and the tokens they are continued with."""
    n = case["seqs"]
    lens = [max(1, case["prompt"] * (4 - 3 * i // max(1, n - 1)) // 4) for i in range(n)]
    return ([_tokens(seed, f"request{i}", k, _VOCAB) for i, k in enumerate(lens)],
            [_tokens(seed, f"step{i}", n, _VOCAB) for i in range(case["steps"])])


def prepare(case, seed):
    from kuiperllama_amd import binfmt, checkpoint
    from kuiperllama_amd.model import KuiperModel
    kind = case["kind"]
    if kind == "operators":
        return _prepare_operators(case, seed)
    if kind == "bin":
        g = _Geom(case["model"])
        spec = binfmt.ModelSpec(g.dim, g.hidden, g.layers, g.heads, g.kv_heads, g.vocab, g.rows, g.tied,
                                binfmt.FAMILY_QWEN2 if g.bias else binfmt.FAMILY_LLAMA, g.quant, _GROUP,
                                binfmt.ROPE_HALF if g.half else binfmt.ROPE_INTERLEAVED, g.theta, g.eps, case["model"])
        table, total = binfmt.layout(spec)
        # the bytes behind the header start on a page, as in the arena that a file is loaded into
        buf = torch.zeros(total + 4096, dtype=torch.uint8, device="cuda")
        lead = -(buf.data_ptr() + spec.header_bytes()) % 4096
        img = buf[lead: lead + total]
        head = [g.dim, g.hidden, g.layers, g.heads, g.kv_heads, g.vocab if g.tied else -g.vocab, g.rows]
        head += [_GROUP] if g.quant else []
        img[: 4 * len(head)] = torch.frombuffer(bytearray(struct.pack("<%di" % len(head), *head)), dtype=torch.uint8).cuda()
        scale = None
        for e in table:
            dst = img[e.offset: e.offset + e.nbytes]
            if e.name.startswith("freqs"):
                continue  # recomputed by the loader
            if e.dtype == "i8":
                q, scale = _quantised(_bin_weight(g, seed, e.name, e.shape))
                dst.copy_(q.reshape(-1).view(torch.uint8))
            elif e.name.endswith(".scales"):
                dst.copy_(scale.view(torch.uint8))
            else:
                dst.copy_(_bin_weight(g, seed, e.name, e.shape).reshape(-1).view(torch.uint8))
        m = KuiperModel.from_device_image(img, spec)
        return {"kind": "bin", "model": m, "prompt": _tokens(seed, "prompt", case["prompt"], g.vocab), "steps": case["steps"]}
    cfg = _layers_config(case)
    tensors = {k: _layer_weight(cfg, seed, k, s).view(torch.int16).cpu().numpy().view(np.uint16)
               for k, s in checkpoint.tensor_shapes(cfg).items()}
    m = KuiperModel.from_tensors(cfg, checkpoint.safetensors_image(tensors), max_seq_len=_POSITIONS, dtype=case["dtype"],
                                 max_seqs=case.get("seqs", 1))
    state = {"kind": kind, "model": m, "steps": case.get("steps", 0)}
    if kind == "serve":
        state["prompts"], state["given"] = _requests(case, seed)
    else:
        state["prompt"] = _tokens(seed, "prompt", case["prompt"], _VOCAB)
    return state


def _prepare_operators(case, seed):
    from kuiperllama_amd import ops
    g, pos = _Geom(case["model"]), case["position"]
    z = lambda *s: torch.zeros(s, device="cuda")
    w = {n: _bin_weight(g, seed, n + ".0", s) for n, s in g.mats.items()}
    if g.quant:
        w = {n: _quantised(v) for n, v in w.items()}
    w.update({n: _bin_weight(g, seed, n + ".0", (g.dim,)) for n in ("att_norm", "ffn_norm")})
    kc, vc = z(g.rows, g.kv), z(g.rows, g.kv)
    kc[:pos], vc[:pos] = _normal(seed, "keys", (pos, g.kv)), _normal(seed, "values", (pos, g.kv))
    sin, cos = z(g.rows, g.hs), z(g.rows, g.hs)
    ops.sincos_cache(g.hs, g.rows, g.theta, sin, cos)
    torch.cuda.synchronize()
    return {"kind": "operators", "g": g, "pos": pos, "w": w, "x": _normal(seed, "x", (g.dim,)), "kc": kc, "vc": vc,
            "sin": sin, "cos": cos, "score": z(g.heads, g.rows), "xn": z(g.dim), "q": z(g.dim), "att": z(g.dim),
            "y": z(g.dim), "x1": z(g.dim), "h1": z(g.hidden), "h3": z(g.hidden), "h": z(g.hidden), "out": z(g.dim)}


# ---- one pass ----------------------------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "operators":
        return _run_operators(state)
    m = state["model"]
    if kind in ("bin", "generate"):
        words, _ = m.generate(state["prompt"], state["steps"])
        return {"tokens": np.array(words[len(state["prompt"]) - 1:], np.int32), "logits": m.logits()}
    if kind == "prompt":
        seq = m.open_seq()
        p = state["prompt"]
        out = m.forward([(seq, p, [len(p) - 1])])
        m.close_seq(seq)
        return out
    seqs = [m.open_seq() for _ in state["prompts"]]
    out = [m.forward([(s, p, [len(p) - 1]) for s, p in zip(seqs, state["prompts"])])]
    for given in state["given"]:
        out.append(m.forward([(s, [t], [0]) for s, t in zip(seqs, given)]))
    for s in seqs:
        m.close_seq(s)
    return out


def _run_operators(s):
    from kuiperllama_amd import ops
    g, pos, w, k, v = s["g"], s["pos"], s["w"], s["kc"][s["pos"]], s["vc"][s["pos"]]

    def matmul(x, name, out):
        if g.quant:
            ops.matmul_q8(x, w[name][0], w[name][1], _GROUP, out)
        else:
            ops.matmul(x, w[name], out)

    ops.rmsnorm(s["x"], w["att_norm"], s["xn"], g.eps)
    matmul(s["xn"], "wq", s["q"])
    matmul(s["xn"], "wk", k)
    matmul(s["xn"], "wv", v)
    ops.rope(s["q"], k, pos, s["sin"], s["cos"], g.hs, ops.ROPE_HALF if g.half else ops.ROPE_INTERLEAVED)
    ops.mha(pos, g.heads, 0, g.rows, g.kv, g.heads // g.kv_heads, g.hs, s["att"], s["q"], s["score"], s["kc"], s["vc"])
    matmul(s["att"], "wo", s["y"])
    ops.add(s["x"], s["y"], s["x1"])
    ops.rmsnorm(s["x1"], w["ffn_norm"], s["xn"], g.eps)
    matmul(s["xn"], "w1", s["h1"])
    matmul(s["xn"], "w3", s["h3"])
    ops.swiglu(s["h1"], s["h3"], s["h"])
    matmul(s["h"], "w2", s["y"])
    ops.add(s["x1"], s["y"], s["out"])
    return {"x": s["out"], "key": k, "value": v}


# ---- the work that a pass cannot do without ----------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("bin", "operators"):
        g = _Geom(case["model"])
        qkv = (g.dim + 2 * g.kv) * g.dim
        layer = qkv + g.dim * g.dim + 3 * g.dim * g.hidden
        if kind == "operators":
            rows = case["position"] + 1
            return {"bytes": g.weight_bytes(layer) + 8 * g.kv * rows, "flops": 2 * layer + 4 * g.dim * rows}
        head, n = g.vocab * g.dim, case["steps"]
        fed = case["prompt"] - 1  # tokens whose logits nobody asks for: of the last layer only their keys and values
        fed = fed if fed < n else 0
        new = n - fed
        nbytes = new * g.weight_bytes(layer * g.layers + head) + 4 * g.vocab
        nbytes += sum(8 * g.kv * g.layers * (p + 1) for p in range(fed, n))
        flops = 2 * new * (layer * g.layers + head) + sum(4 * g.dim * g.layers * (p + 1) for p in range(fed, n))
        if fed:
            flops += 2 * fed * (layer * (g.layers - 1) + 2 * g.kv * g.dim) + 2 * g.dim * (g.layers - 1) * fed * (fed + 1)
            nbytes += 8 * g.kv * g.layers * fed  # their weights are read once with those of the first new token at best
        return {"bytes": nbytes, "flops": flops}
    cfg = _layers_config(case)
    el = 2 if case["dtype"] == "bfloat16" else 4
    if kind == "prompt":
        batches = [(1, [(0, case["prompt"])])]
    elif kind == "generate":
        fed = case["prompt"] - 1
        batches = [(0, [(0, fed)])] if fed else []
        batches += [(1, [(p, 1)]) for p in range(fed, case["steps"])]
    else:
        lens = [len(p) for p in _requests(case, 0)[0]]
        batches = [(len(lens), [(0, n) for n in lens])]
        batches += [(len(lens), [(n + i, 1) for n in lens]) for i in range(case["steps"])]
    nbytes = flops = 0.0
    for want, segs in batches:
        T = sum(n for _, n in segs)
        for layer in cfg["layers"]:
            fixed, used = _layer_sizes(cfg, layer, T)
            nbytes += el * used
            flops += 2 * T * fixed
            m = layer["mixer"]
            if layer["type"] == "mamba1":
                flops += 7 * T * m["inner"] * m["state"]
                nbytes += len(segs) * 8 * m["inner"] * m["state"]
                continue
            size = m.get("mask", {}).get("size", 1 << 30)
            row = m["kv_rank"] + m["rot_dim"] if "kv_rank" in m else m["kv_heads"] * (m["dim"] + m["vdim"])
            per = 2 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"])
            for p0, n in segs:
                if layer["type"] == "attention_2":
                    keys = sum(p % size + 1 for p in range(p0, p0 + n))
                else:
                    keys = sum(min(p + 1, size) for p in range(p0, p0 + n))
                flops += per * keys
                nbytes += el * row * (n + min(p0, size))
        nbytes += want * cfg["vocab"] * 4 + (el * cfg["vocab"] * cfg["width"] if want else 0)
        flops += 2 * want * cfg["vocab"] * cfg["width"]
    return {"bytes": nbytes, "flops": flops}


def _layer_sizes(cfg, layer, T):
    """Weights that a token of the layer is multiplied with, and weights that T tokens read at least once (random routes)."""
    W, m, f = cfg["width"], layer["mixer"], layer["mlp"]
    if layer["type"] == "mamba1":
        mix = 3 * m["inner"] * W + m["inner"] * (2 * m["dt_rank"] + 2 * m["state"] + m["conv"])
    elif layer["type"] == "latent_attention":
        H = m["heads"]
        mix = (W * (m["q_rank"] + m["kv_rank"] + m["rot_dim"]) + m["q_rank"] * H * (m["dim"] + m["rot_dim"]) +
               m["kv_rank"] * H * (m["dim"] + m["vdim"]) + W * H * m["vdim"])
    else:
        gate = layer["type"] == "attention_2"
        mix = W * (m["heads"] * (m["dim"] + m["vdim"] * (2 if gate else 1)) + m["kv_heads"] * (m["dim"] + m["vdim"]))
    if f["kind"] == "dense":
        return mix + 3 * W * f["ff"], mix + 3 * W * f["ff"]
    r = f["router"]
    n_out = r["experts"] + r.get("identity", 0)
    rest = W * n_out + (3 * W * f["shared"]["ff"] if f.get("shared") else 0)
    one = 3 * W * f["expert"]["ff"]
    share = r["experts"] / n_out
    met = r["experts"] * (1.0 - (1.0 - r["top"] / n_out) ** T)
    return mix + rest + one * r["top"] * share, mix + rest + one * met


# ---- how far two correct implementations lie apart ---------------------------------------------------------------------
def tolerance(case):
    """About four times the distance of the paths from their 64-bit results: 3.4e-3 in bf16 (a token whose last expert is
    nearly a tie may go to another one), 1.6e-6 in fp32 over a whole model, 6.7e-6 where int8 groups are summed in fp32,
    1.4e-7 over one layer."""
    if case["kind"] == "operators":
        rel = 1e-6
    elif case.get("dtype") == "bfloat16":
        rel = 2e-2
    else:
        rel = 3e-5 if case.get("model") == "llama2-7b-int8" else 8e-6
    return {"rel": rel, "max": 10 * rel, "differ": 0.0}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------
def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "operators":
            return _exact_operators(case, seed)
        if case["kind"] == "bin":
            return _exact_greedy(_Exact64(_Geom(case["model"]), seed), _tokens(seed, "prompt", case["prompt"], _BIN[case["model"]][5]),
                                 case["steps"])
        cfg = _layers_config(case)
        if case["kind"] == "prompt":
            p = _tokens(seed, "prompt", case["prompt"], _VOCAB)
            return _Layers64(cfg, seed)(p)[-1:].cpu().numpy()
        if case["kind"] == "generate":
            return _exact_greedy(_Layers64(cfg, seed), _tokens(seed, "prompt", case["prompt"], _VOCAB), case["steps"])
        prompts, given = _requests(case, seed)
        cols = []
        for i, p in enumerate(prompts):
            z = _Layers64(cfg, seed)(p + [t[i] for t in given])
            cols.append(z[len(p) - 1:])
        return [torch.stack([c[j] for c in cols]).cpu().numpy() for j in range(case["steps"] + 1)]


def _exact_greedy(model, prompt, steps):
    fed = prompt[: min(len(prompt), steps)]
    z = model(fed)[-1]
    words = [int(z.argmax())] if len(fed) == len(prompt) else []
    for _ in range(len(fed), steps):
        z = model([words[-1]])[-1]
        words.append(int(z.argmax()))
    return {"tokens": np.array(words, np.int32), "logits": z.cpu().numpy()}


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _angles(hs, theta, pos):
    """The format's rotation table is defined in 32 bits: theta^(-d/hs) and its product with the position."""
    p = (np.float64(np.float32(theta)) ** np.float64(np.arange(0, hs, 2, dtype=np.float32) / np.float32(hs))).astype(np.float32)
    f = np.float32(1.0) / p
    return torch.from_numpy((pos.astype(np.float32)[:, None] * f[None, :]).astype(np.float64)).cuda()


def _rotate(v, ang, half):
    """v [T, heads, hs]"""
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    n = v.shape[-1] // 2
    a, b = (v[..., :n], v[..., n:]) if half else (v[..., 0::2], v[..., 1::2])
    x, y = a * c - b * s, a * s + b * c
    return torch.cat([x, y], -1) if half else torch.stack([x, y], -1).flatten(-2)


def _attend64(q, k, v, seen, scale, bias=None, extra=None):
    """q [T, H, d], k, v [N, G, d]; seen [T, N]; extra: one more score per head in the denominator (tensor [H])."""
    H, G = q.shape[1], k.shape[1]
    out = []
    for h in range(H):
        s = q[:, h] @ k[:, h * G // H].T * scale
        if bias is not None:
            s = s + bias[h]
        s = s.masked_fill(~seen, -math.inf)
        if extra is not None:
            s = torch.cat([s, extra[h].expand(len(s), 1)], 1)
        p = torch.softmax(s, -1)
        out.append(p[:, : k.shape[0]] @ v[:, h * G // H])
    return torch.stack(out, 1).flatten(1)


class _Exact64:
    """A .bin model; calls append tokens and return the logits of the last."""

    def __init__(self, g, seed):
        self.g, self.seed, self.n, self.w = g, seed, 0, {}
        self.k, self.v = [None] * g.layers, [None] * g.layers

    def mat(self, name, shape, quant=None):
        if name not in self.w:
            w = _bin_weight(self.g, self.seed, name, shape)
            self.w[name] = _quantised(w) if (self.g.quant if quant is None else quant) else w
        w = self.w[name]
        if isinstance(w, tuple):
            return (w[0].double().reshape(-1, _GROUP) * w[1].double()[:, None]).reshape(shape)
        return w.double()

    def layer(self, l, x, pos):
        g = self.g
        w = lambda n: self.mat(f"{n}.{l}", g.mats[n])
        vec = lambda n, k: self.mat(f"{n}.{l}", (k,), False)
        h = _rms64(x, vec("att_norm", g.dim), g.eps)
        q, k, v = h @ w("wq").T, h @ w("wk").T, h @ w("wv").T
        if g.bias:
            q, k, v = q + vec("bq", g.dim), k + vec("bk", g.kv), v + vec("bv", g.kv)
        ang = _angles(g.hs, g.theta, pos)
        q = _rotate(q.reshape(len(x), g.heads, g.hs), ang, g.half)
        k = _rotate(k.reshape(len(x), g.kv_heads, g.hs), ang, g.half)
        v = v.reshape(len(x), g.kv_heads, g.hs)
        new = (k, v)
        if self.k[l] is not None:
            k, v = torch.cat([self.k[l], k]), torch.cat([self.v[l], v])
        self.k[l], self.v[l] = k, v
        p = torch.from_numpy(pos).cuda()
        seen = torch.arange(k.shape[0], device="cuda")[None, :] <= p[:, None]
        x = x + _attend64(q, k, v, seen, g.hs ** -0.5) @ w("wo").T
        h = _rms64(x, vec("ffn_norm", g.dim), g.eps)
        return x + (torch.nn.functional.silu(h @ w("w1").T) * (h @ w("w3").T)) @ w("w2").T, new

    def __call__(self, tokens):
        g = self.g
        emb = self.mat("tok_emb", (g.vocab, g.dim), False)
        x, pos = emb[torch.tensor(tokens, device="cuda")], np.arange(self.n, self.n + len(tokens))
        if not g.tied:
            del emb
        self.n += len(tokens)
        for l in range(g.layers):
            x, _ = self.layer(l, x, pos)
        x = _rms64(x[-1:], self.mat("final_norm", (g.dim,), False), g.eps)
        return x @ (emb if g.tied else self.mat("wcls", (g.vocab, g.dim))).T


def _exact_operators(case, seed):
    g, pos = _Geom(case["model"]), case["position"]
    g.bias = False
    e = _Exact64(g, seed)
    rows = lambda n: _normal(seed, n, (pos, g.kv)).double().reshape(pos, g.kv_heads, g.hs)
    e.k[0], e.v[0] = rows("keys"), rows("values")
    x, (k, v) = e.layer(0, _normal(seed, "x", (g.dim,)).double()[None], np.array([pos]))
    return {"x": x[0].cpu().numpy(), "key": k.flatten().cpu().numpy(), "value": v.flatten().cpu().numpy()}


class _Layers64:
    """A layer-list model.  Calls append tokens (the whole sequence is run again) and return all logits."""

    def __init__(self, cfg, seed):
        self.c, self.seed, self.tokens = cfg, seed, []

    def w(self, name, *shape):
        return _layer_weight(self.c, self.seed, name, shape).double()

    def __call__(self, tokens):
        c, W = self.c, self.c["width"]
        self.tokens = self.tokens + list(tokens)
        T, eps, gufanex = len(self.tokens), c["norm"]["eps"], c["architecture"] == "Gufanex"
        x = self.w("embed", c["vocab"], W)[torch.tensor(self.tokens, device="cuda")]
        if not gufanex:
            x = x * c["embedding"]["scale"] + self.w("pos", c["max_positions"], W)[:T]

        def norm(name, v):
            if not gufanex:
                return _rms64(v, 1.0 + self.w(name, W), eps)
            return torch.nn.functional.layer_norm(v, (W,), self.w(name, W), self.w(name + ".b", W), eps)

        mixers = {"mamba1": self.mamba, "latent_attention": self.latent, "attention": self.heads, "attention_2": self.heads}
        for i, l in enumerate(c["layers"]):
            h = norm(f"l{i}.norm1", x)
            d = mixers[l["type"]](f"l{i}.mix", l["mixer"], h, eps)
            d = d + self.feed(f"l{i}.mlp", l["mlp"], norm(f"l{i}.norm2", x) if gufanex else h)
            x = x + d * c.get("residual_mult", 1.0)
        z = norm("final.norm", x) @ self.w("head", c["vocab"], W).T
        cap = c.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z

    def mamba(self, p, m, h, eps):
        W, I, N, r, taps = self.c["width"], m["inner"], m["state"], m["dt_rank"], m["conv"]
        xz = h @ self.w(p + ".in", 2 * I, W).T
        x, z = xz[:, :I], xz[:, I:]
        cw, T = self.w(p + ".conv", I, taps), len(h)
        pad = torch.cat([x.new_zeros(taps - 1, I), x])
        x = self.w(p + ".conv.b", I) + sum(pad[k: k + T] * cw[:, k] for k in range(taps))
        x = torch.nn.functional.silu(x)
        dbc = x @ self.w(p + ".x", r + 2 * N, I).T
        dt = dbc[:, :r] @ self.w(p + ".dt", I, r).T + self.w(p + ".dt.b", I)
        dt = torch.logaddexp(dt, torch.zeros_like(dt))
        A, B, C = -torch.exp(self.w(p + ".A_log", I, N)), dbc[:, r: r + N], dbc[:, r + N:]
        S, y = x.new_zeros(I, N), torch.empty_like(x)
        dx = dt * x
        for t in range(T):
            S = torch.exp(dt[t][:, None] * A) * S + dx[t][:, None] * B[t]
            y[t] = S @ C[t]
        y = y + self.w(p + ".D", I) * x
        return (y * torch.nn.functional.silu(z)) @ self.w(p + ".o", W, I).T

    def latent(self, p, m, h, eps):
        W, H, dn, dr, dv, R, Q = self.c["width"], m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
        T = len(h)
        q = (_rms64(h @ self.w(p + ".dq", Q, W).T, self.w(p + ".dq.norm", Q), eps) @ self.w(p + ".uq", H * (dn + dr), Q).T)
        q = q.reshape(T, H, dn + dr)
        kv = h @ self.w(p + ".dkv", R + dr, W).T
        c = _rms64(kv[:, :R], self.w(p + ".dkv.norm", R), eps)
        n = m["rot"]["dims"]
        f = m["rot"]["base"] ** (-torch.arange(0, n, 2, device="cuda").double() / n)
        ang = torch.arange(T, device="cuda").double()[:, None] * f[None, :]

        def turn(v):
            return torch.cat([_rotate(v[..., :n], ang, False), v[..., n:]], -1)

        kr = turn(kv[:, None, R:]).expand(T, H, dr)
        k = torch.cat([(c @ self.w(p + ".uk", H * dn, R).T).reshape(T, H, dn), kr], -1)
        v = (c @ self.w(p + ".uv", H * dv, R).T).reshape(T, H, dv)
        q = torch.cat([q[..., :dn], turn(q[..., dn:])], -1)
        t = torch.arange(T, device="cuda")
        a = _attend64(q, k, v, t[None, :] <= t[:, None], m["scale"], extra=self.w(p + ".sink", H))
        return a @ self.w(p + ".o", W, H * dv).T

    def heads(self, p, m, h, eps):
        W, H, G, dk, dv, T = self.c["width"], m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
        chunk = "bias_max" not in m

        def proj(n, heads, d):
            y = h @ self.w(f"{p}.{n}", heads * d, W).T
            return (y + self.w(f"{p}.{n}.b", heads * d) if chunk else y).reshape(T, heads, d)

        q = _rms64(proj("q", H, dk), self.w(p + ".q.norm", dk), eps)
        k = _rms64(proj("k", G, dk), self.w(p + ".k.norm", dk), eps)
        v = proj("v", G, dv)
        t = torch.arange(T, device="cuda")
        d, size = t[:, None] - t[None, :], m["mask"]["size"]
        if chunk:
            seen = (d >= 0) & (t[:, None] // size == t[None, :] // size)
            a = _attend64(q, k, v, seen, m["scale"], extra=torch.zeros(H, dtype=torch.float64, device="cuda"))
            a = a * torch.sigmoid(h @ self.w(p + ".g", H * dv, W).T)
            return a @ self.w(p + ".o", W, H * dv).T + self.w(p + ".o.b", W)
        rows = 32
        rel, half = self.w(p + ".rel", rows, H), rows // 2
        n = np.arange(T)
        far = np.log(np.maximum(n, 1) / half) / math.log(m["bias_max"] / half) * (rows - half)
        near = np.round(far)
        far = np.where(np.abs(far - near) < 1e-9, near, np.floor(far))
        row = torch.from_numpy(np.where(n < half, n, np.minimum(rows - 1, half + far)).astype(np.int64)).cuda()
        bias = rel[row[d.clamp(min=0)]].permute(2, 0, 1)
        a = _attend64(q, k, v, (d >= 0) & (d < size), m["scale"], bias=bias)
        return a @ self.w(p + ".o", W, H * dv).T

    def unit(self, p, ff, h, limit=None):
        W = self.c["width"]
        g, u = h @ self.w(p + ".gate", ff, W).T, h @ self.w(p + ".up", ff, W).T
        if limit is None:
            y = torch.nn.functional.silu(g) * u
        else:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            y = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        return y @ self.w(p + ".down", W, ff).T

    def feed(self, p, f, h):
        W = self.c["width"]
        if f["kind"] == "dense":
            return self.unit(p, f["ff"], h)
        E, top = f["router"]["experts"], f["router"]["top"]
        n_out = E + f["router"].get("identity", 0)
        z = h @ self.w(p + ".router", n_out, W).T
        if "limit" in f["expert"]:
            c, ids = torch.topk(z, top, -1)
            g = torch.softmax(c, -1)
        else:
            s = torch.softmax(z, -1)
            ids = torch.topk(s + self.w(p + ".correction", n_out), top, -1).indices
            g = s.gather(-1, ids)
        weight = torch.zeros_like(z).scatter(-1, ids, g)
        out = weight[:, E:].sum(-1, keepdim=True) * h
        for e in range(E):
            rows = (ids == e).any(-1).nonzero()[:, 0]
            if len(rows):
                y = self.unit(f"{p}.e{e}", f["expert"]["ff"], h[rows], f["expert"].get("limit"))
                out[rows] += weight[rows, e, None] * y
        if f.get("shared"):
            gate = torch.sigmoid(h @ self.w(p + ".shared.sg", 1, W).T)
            out = out + gate * self.unit(p + ".shared", f["shared"]["ff"], h)
        return out
