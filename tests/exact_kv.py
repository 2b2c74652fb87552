"""K and V rows of a .bin model in 64 bits, and how far a pass is from them."""
import numpy as np
import torch

from kuiperllama_amd import binfmt


def tensors(img, spec):
    return {e.name: binfmt.tensor_from_image(img, e) for e in binfmt.layout(spec)[0]}


def _weights(img, spec):
    w, t = {}, tensors(img, spec)
    for n, v in t.items():
        if n.startswith("freqs") or n.endswith(".scales"):
            continue
        d = v.detach().cpu().double()
        if v.dtype == torch.int8:
            d = (d.reshape(-1, spec.group_size) * t[n + ".scales"].cpu().double()[:, None]).reshape(v.shape)
        w[n] = d
    return w


def _rotate(x, spec, pos):
    """x [T, heads * head_size]; the angles are 32-bit numbers in the format."""
    hs = spec.head_size
    p = np.float64(np.float32(spec.rope_theta)) ** np.float64(np.arange(0, hs, 2, dtype=np.float32) / np.float32(hs))
    f = np.float32(1.0) / p.astype(np.float32)
    ang = torch.from_numpy((pos.astype(np.float32)[:, None] * f[None, :]).astype(np.float64))[:, None]
    v = x.reshape(len(x), -1, hs)
    half = spec.rope_mode == binfmt.ROPE_HALF
    a, b = (v[..., : hs // 2], v[..., hs // 2:]) if half else (v[..., 0::2], v[..., 1::2])
    p, q = a * torch.cos(ang) - b * torch.sin(ang), a * torch.sin(ang) + b * torch.cos(ang)
    return (torch.cat([p, q], -1) if half else torch.stack([p, q], -1).flatten(-2)).reshape(x.shape)


def rows(img, spec, toks, front=None, logits=None):
    """[(K, V)] per layer of `toks` behind the cache rows front[layer] = (K, V).  logits: a list that gets the last token's."""
    w, hs, mul = _weights(img, spec), spec.head_size, spec.kv_mul
    old = 0 if front is None else len(front[0][0])
    pos, out = np.arange(old, old + len(toks)), []
    x = w["tok_emb"][torch.tensor(toks)]
    norm = lambda v, g: v / torch.sqrt((v * v).mean(-1, keepdim=True) + spec.rms_eps) * g
    for l in range(spec.n_layers):
        h = norm(x, w[f"att_norm.{l}"])
        q, k, v = (h @ w[f"{n}.{l}"].T + w.get(f"b{n[1]}.{l}", 0.0) for n in ("wq", "wk", "wv"))
        q, k = _rotate(q, spec, pos), _rotate(k, spec, pos)
        out.append((k.numpy(), v.numpy()))
        if front is not None:
            k, v = (torch.cat([torch.from_numpy(f).double(), n]) for f, n in zip(front[l], (k, v)))
        seen = torch.arange(len(k))[None, :] <= torch.from_numpy(pos)[:, None]
        att = []
        for i in range(spec.n_heads):
            g = slice(i // mul * hs, i // mul * hs + hs)
            s = (q[:, i * hs: i * hs + hs] @ k[:, g].T / hs ** 0.5).masked_fill(~seen, -torch.inf)
            att.append(torch.softmax(s, -1) @ v[:, g])
        x = x + torch.cat(att, 1) @ w[f"wo.{l}"].T
        h = norm(x, w[f"ffn_norm.{l}"])
        x = x + (torch.nn.functional.silu(h @ w[f"w1.{l}"].T) * (h @ w[f"w3.{l}"].T)) @ w[f"w2.{l}"].T
    if logits is not None:
        logits.append((norm(x[-1], w["final_norm"]) @ w["tok_emb" if spec.shared_classifier else "wcls"].T).numpy())
    return out


def error(got, want):
    """Largest over the columns of the rms of the difference relative to the rms of the column."""
    d = np.sqrt(((got.astype(np.float64) - want) ** 2).mean(0))
    return float((d / np.maximum(np.sqrt((want ** 2).mean(0)), 1e-300)).max())
