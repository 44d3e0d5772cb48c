"""The work that programs have this package do, as cases that can be timed.

Every case is one of eight paths through the public entry points, each named after what calls it:

  attention   one attention call of an encoder layer, or a causal one (embedding, reranking, speech)
  step        the attention of one decoder step over a cache that holds every layer's heads
  prefill     a Qwen3 layer's way to its attention: residual add + RMSNorm, projection, prologue, causal attention
  decode      the same for one new token a sequence, over a cache with the token's own row appended
  local       a ModernBERT layer's: LayerNorm, projection with the rope in its store, packed attention in a window
  prologue    the split of a fused projection into normalised, rotated heads, by itself
  norm        a row norm, with or without the residual add
  projection  a fused projection, with a bias or with the rope

Sizes are those of the models that the tests and the benchmark name, over the batches and lengths that
services see: one short query up to a full batch of long documents.
"""
import math

import torch

import svod_amd
from svod_amd import Attn, Cache, KeyMask, Linear, Qkv, Rotary
from svod_amd.workloads import rope_table

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
EPS = 1e-6

# (hidden size, query heads, KV heads, head size) of a layer's attention.
QWEN3 = (1024, 16, 8, 128)
MODERNBERT = (768, 12, 12, 64)
BGE_M3 = (1024, 16, 16, 64)
LAYERS = {"qwen3": QWEN3, "modernbert": MODERNBERT, "bge_m3": BGE_M3}


def listed():
    return [
        # A search query embedded by itself, as it comes in: BGE-M3's heads over a handful of tokens.  Latency.
        {"name": "query_attention", "path": "attention", "batch": 1, "seq": 19, "heads": 16, "kv_heads": 16,
         "head_dim": 64, "causal": False, "mask": "bool", "least": 1.0, "dtype": "bf16"},
        # BGE-M3 over a full batch of passages, padded to the longest, with the [B, Tk] mask the model passes.
        {"name": "passages_attention", "path": "attention", "batch": 32, "seq": 512, "heads": 16, "kv_heads": 16,
         "head_dim": 64, "causal": False, "mask": "bool", "least": 0.125, "dtype": "bf16"},
        # A middling batch at a length that is no multiple of anything, in f16, with key lengths.
        {"name": "ragged_attention_f16", "path": "attention", "batch": 9, "seq": 333, "heads": 12, "kv_heads": 12,
         "head_dim": 64, "causal": False, "mask": "lens", "least": 0.3, "dtype": "f16"},
        # Whisper-large-v3's encoder: 30 s of audio are 1500 frames, nothing masked.
        {"name": "speech_attention", "path": "attention", "batch": 16, "seq": 1500, "heads": 20, "kv_heads": 20,
         "head_dim": 64, "causal": False, "mask": "none", "least": 1.0, "dtype": "bf16"},
        # A reranker's pair of long documents: the largest single call.
        {"name": "documents_attention", "path": "attention", "batch": 2, "seq": 8192, "heads": 16, "kv_heads": 16,
         "head_dim": 64, "causal": False, "mask": "lens", "least": 0.6, "dtype": "bf16"},
        # Whisper's decoder, one token a lane: cross-attention over the encoder's keys in a cache of 32 layers.
        {"name": "speech_step", "path": "step", "batch": 16, "keys": 1500, "heads": 20, "kv_heads": 20, "head_dim": 64,
         "layers": 32, "least": 1.0, "dtype": "bf16"},
        # Qwen3-Embedding over a batch of passages: the attention half of a layer.
        {"name": "passages_prefill", "path": "prefill", "batch": 8, "seq": 2048, "least": 0.25, "dtype": "bf16"},
        # A single instruction-and-query through the same layer: every launch is short.
        {"name": "query_prefill", "path": "prefill", "batch": 1, "seq": 45, "least": 1.0, "dtype": "bf16"},
        # Generating with the Qwen3 layer: 16 sequences, a token each, some 2000 cached keys.
        {"name": "tokens_decode", "path": "decode", "batch": 16, "keys": 2100, "layers": 2, "least": 0.25, "dtype": "bf16"},
        # ModernBERT's local layers over passages of odd length.
        {"name": "passages_local", "path": "local", "batch": 8, "seq": 777, "window": 64, "least": 0.2, "dtype": "bf16"},
        # The residual add + RMSNorm between layers of hidden size 2048, over a full batch.
        {"name": "batch_norm_rows", "path": "norm", "form": "add_rms_norm", "tokens": 16384, "width": 2048, "dtype": "bf16"},
        # BGE-M3's fused projection with its bias over the tokens of a middling batch.
        {"name": "batch_projection", "path": "projection", "layer": "bge_m3", "batch": 8, "seq": 500, "dtype": "bf16"},
    ]


def _spread(rng, low, high):
    """A whole number from `low` to `high`, even over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _batch(rng):
    """A batch of sequences, up to a full one: (how many, how long)."""
    tokens = _spread(rng, 8, 16384)
    batch = _spread(rng, 1, max(1, min(32, tokens // 8)))
    return batch, max(8, min(4096, tokens // batch))


def draw(rng):
    path = rng.choice(["attention"] * 4 + ["step"] * 2 + ["prefill"] * 2 + ["decode"] * 2 + ["local"] * 2 +
                      ["prologue", "norm", "projection"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    least = round(rng.uniform(0.1, 1.0), 3)
    if path == "attention":
        heads, kv_heads, head_dim, causal = rng.choice([(16, 16, 64, False), (12, 12, 64, False), (20, 20, 64, False),
                                                        (16, 8, 128, True)])
        seq = _spread(rng, 8, 8192)
        pairs = 9 * 2 * 16 * 8192 * 8192 * 64 // (10 * heads * head_dim)  # what the largest listed call sees
        batch = _spread(rng, 1, max(1, min(64, pairs // (seq * seq), 32768 // seq)))
        mask = "lens" if causal else rng.choice(["lens", "bool", "none"])
        return {"path": path, "batch": batch, "seq": seq, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
                "causal": causal, "mask": mask, "least": 1.0 if mask == "none" else least, "dtype": dtype}
    if path == "step":
        heads, kv_heads, head_dim = rng.choice([(20, 20, 64), (16, 16, 64), (32, 32, 64), (16, 8, 128)])
        keys = _spread(rng, 32, 8192)
        batch = _spread(rng, 1, max(1, min(64, 65536 // keys)))
        return {"path": path, "batch": batch, "keys": keys, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
                "layers": rng.choice([1, 4, 8]), "least": rng.choice([1.0, least]), "dtype": dtype}
    if path in ("prefill", "local"):
        batch, seq = _batch(rng)
        case = {"path": path, "batch": batch, "seq": seq, "least": least, "dtype": dtype}
        if path == "local":
            case["window"] = rng.choice([64, 64, 0])  # every third layer sees every key
        return case
    if path == "decode":
        keys = _spread(rng, 32, 8192)
        return {"path": path, "batch": _spread(rng, 1, max(1, min(64, 65536 // keys))), "keys": keys,
                "layers": rng.choice([1, 2, 4]), "least": least, "dtype": dtype}
    if path == "norm":
        form, width = rng.choice([("rms_norm", 1024), ("add_rms_norm", 1024), ("add_rms_norm", 2048), ("layer_norm", 768),
                                  ("add_layer_norm", 768), ("add_layer_norm", 1024)])
        return {"path": path, "form": form, "tokens": _spread(rng, 1, 16384), "width": width, "dtype": dtype}
    # A decoder step has a token a sequence, everything else whole sequences.
    batch, seq = (_spread(rng, 1, 64), 1) if rng.random() < 0.25 else _batch(rng)
    case = {"path": path, "batch": batch, "seq": seq, "dtype": dtype}
    if path == "projection":
        case["layer"] = rng.choice(sorted(LAYERS))
    return case


# ---- what a program holds before the call.

class _Maker:
    """Tensors of one case, from its seed alone."""

    def __init__(self, case, seed):
        self.device = torch.device("cuda")
        self.dtype = DTYPES[case["dtype"]]
        self.g = torch.Generator(device=self.device).manual_seed(seed)

    def normal(self, *shape, sigma=1.0):
        x = torch.empty(shape, dtype=self.dtype, device=self.device)
        return x.normal_(0.0, sigma, generator=self.g)

    def gain(self, n):
        return (0.8 + 0.4 * torch.rand(n, generator=self.g, device=self.device)).to(self.dtype)

    def counts(self, n, most, least):
        """`n` key counts from `least * most` to `most`; a padded batch is as long as its longest row."""
        low = max(1, int(least * most))
        c = torch.randint(low, most + 1, (n,), generator=self.g, device=self.device, dtype=torch.int32)
        c[torch.randint(0, n, (1,), generator=self.g, device=self.device)] = most
        return c

    def rope(self, seq, head_dim, theta=1e6):
        return tuple(a.to(self.dtype).reshape(1, seq, 1, head_dim // 2) for a in rope_table(theta, seq, head_dim, self.device))


def prepare(case, seed):
    m = _Maker(case, seed)
    path = case["path"]
    s = {"path": path}
    if path == "attention":
        b, t, h, hkv, d = (case[k] for k in ("batch", "seq", "heads", "kv_heads", "head_dim"))
        s["q"], s["k"], s["v"] = m.normal(b, t, h, d), m.normal(b, t, hkv, d), m.normal(b, t, hkv, d)
        keys = KeyMask.none()
        if case["mask"] != "none":
            lens = m.counts(b, t, case["least"])
            keys = KeyMask.lens(lens)
            if case["mask"] == "bool":
                keys = KeyMask.bool(torch.arange(t, device=m.device)[None, :] < lens[:, None])
        s["opts"] = Attn(causal=case["causal"], keys=keys)
    elif path == "step":
        b, tk, h, hkv, d, layers = (case[k] for k in ("batch", "keys", "heads", "kv_heads", "head_dim", "layers"))
        s["q"] = m.normal(b, 1, h, d)
        s["k"], s["v"] = m.normal(b, tk, layers * hkv, d), m.normal(b, tk, layers * hkv, d)
        s["opts"] = Attn(keys=KeyMask.lens(m.counts(b, tk, case["least"])), cache=Cache(seed % layers * hkv, hkv))
    elif path in ("prefill", "decode"):
        hidden, h, hkv, d = QWEN3
        b, t = case["batch"], case.get("seq", 1)
        s["x"], s["residual"], s["norm"] = m.normal(b, t, hidden), m.normal(b, t, hidden), m.gain(hidden)
        s["w"] = m.normal((h + 2 * hkv) * d, hidden, sigma=hidden ** -0.5)
        if path == "prefill":
            tables = m.rope(t, d)
            s["opts"] = Attn(causal=True, keys=KeyMask.lens(m.counts(b, t, case["least"])))
        else:
            tk, layers = case["keys"], case["layers"]
            lens = m.counts(b, tk, case["least"])
            # A token stands at the position its sequence has reached: a row of the table for each.
            tables = tuple(a[0, lens.long()].reshape(b, 1, 1, d // 2) for a in m.rope(tk + 1, d))
            s["k"], s["v"] = m.normal(b, tk, layers * hkv, d), m.normal(b, tk, layers * hkv, d)
            # Sequences sit in the cache's rows in the order in which they were admitted.
            s["rows"] = torch.randperm(b, generator=m.g, device=m.device).to(torch.int32)
            s["keys"], s["first"], s["kv_heads"] = KeyMask.lens(lens), seed % layers * hkv, hkv
        s["qkv"] = Qkv(h, hkv, d, m.gain(d), m.gain(d), EPS, tables)
    elif path == "local":
        hidden, h, hkv, d = MODERNBERT
        b, t = case["batch"], case["seq"]
        s["x"], s["norm"], s["heads"] = m.normal(b, t, hidden), m.gain(hidden), (h, hkv)
        s["w"] = m.normal((h + 2 * hkv) * d, hidden, sigma=hidden ** -0.5)
        cos, sin = m.rope(t, d, 1e4)
        s["linear"] = Linear(rope=Rotary(cos, sin, h + hkv, d))
        w = case["window"]
        s["opts"] = Attn(keys=KeyMask.lens(m.counts(b, t, case["least"])), window=(w, w) if w else None)
    elif path == "prologue":
        _, h, hkv, d = QWEN3
        b, t = case["batch"], case["seq"]
        s["x"] = m.normal(b, t, (h + 2 * hkv) * d)
        s["qkv"] = Qkv(h, hkv, d, m.gain(d), m.gain(d), EPS, m.rope(t, d))
    elif path == "norm":
        n, width = case["tokens"], case["width"]
        s["form"], s["x"], s["norm"] = case["form"], m.normal(n, width), m.gain(width)
        if case["form"].startswith("add_"):
            s["residual"] = m.normal(n, width)
        if "layer" in case["form"]:
            s["bias"] = m.normal(width, sigma=0.1)
    else:
        hidden, h, hkv, d = LAYERS[case["layer"]]
        b, t = case["batch"], case["seq"]
        n = (h + 2 * hkv) * d
        s["x"], s["w"] = m.normal(b, t, hidden), m.normal(n, hidden, sigma=hidden ** -0.5)
        if case["layer"] == "modernbert":
            cos, sin = m.rope(t, d, 1e4)
            s["linear"] = Linear(rope=Rotary(cos, sin, h + hkv, d))
        elif case["layer"] == "bge_m3":
            s["linear"] = Linear(bias=m.normal(n, sigma=0.1))
        else:
            s["linear"] = Linear()
    return s


# ---- the call.

def run(state):
    s, path = state, state["path"]
    if path in ("attention", "step"):
        return svod_amd.attention(s["q"], s["k"], s["v"], s["opts"])
    if path == "prefill":
        total, y = svod_amd.add_rms_norm(s["x"], s["residual"], s["norm"], EPS)
        q, k, v = svod_amd.heads(svod_amd.linear(y, s["w"]), s["qkv"])
        return total, k, v, svod_amd.attention(q, k, v, s["opts"])
    if path == "decode":
        total, y = svod_amd.add_rms_norm(s["x"], s["residual"], s["norm"], EPS)
        q, k, v = svod_amd.heads(svod_amd.linear(y, s["w"]), s["qkv"])
        cache = Cache(s["first"], s["kv_heads"], row_map=s["rows"], appended=(k, v))
        return total, k, v, svod_amd.attention(q, s["k"], s["v"], Attn(keys=s["keys"], cache=cache))
    if path == "local":
        y = svod_amd.layer_norm(s["x"], s["norm"], eps=1e-5)
        return svod_amd.attention_packed(svod_amd.linear(y, s["w"], s["linear"]), *s["heads"], s["opts"])
    if path == "prologue":
        return svod_amd.heads(s["x"], s["qkv"])
    if path == "projection":
        return svod_amd.linear(s["x"], s["w"], s["linear"])
    if s["form"] == "rms_norm":
        return svod_amd.rms_norm(s["x"], s["norm"], EPS)
    if s["form"] == "add_rms_norm":
        return svod_amd.add_rms_norm(s["x"], s["residual"], s["norm"], EPS)
    if s["form"] == "layer_norm":
        return svod_amd.layer_norm(s["x"], s["norm"], s["bias"])
    return svod_amd.add_layer_norm(s["x"], s["residual"], s["norm"], s["bias"])


# ---- what a call cannot do without, and how close two correct ones are.

def _lengths(batch, most, least):
    """Key counts evenly spread over the range that prepare() takes them from: their expectation stands for any seed's."""
    low = max(1, int(least * most))
    if batch == 1:
        return [(1.0, most)]
    steps = 16
    spread = (batch - 1) / batch / steps
    return [(1.0 / batch, most)] + [(spread, low + (most - low) * (i + 0.5) / steps) for i in range(steps)]


def _attention_work(batch, t, tk, h, hkv, d, least, causal=False, window=0):
    """Bytes and operations of an attention call: q and o whole, the keys and values that are visible."""
    pairs = keys = 0.0
    for share, n in _lengths(batch, tk, least):
        keys += share * n
        if causal:
            pairs += share * (n * (n + 1) / 2 + (t - n) * n)
        elif window:
            pairs += share * sum(max(0.0, min(n, i + window + 1) - max(0, i - window)) for i in range(t))
        else:
            pairs += share * t * n
    return 2 * batch * (2 * t * h * d + 2 * keys * hkv * d), 4 * d * h * batch * pairs


def work(case):
    path = case["path"]
    if path == "attention":
        b, f = _attention_work(case["batch"], case["seq"], case["seq"], case["heads"], case["kv_heads"], case["head_dim"],
                               case["least"], case["causal"])
        return {"bytes": b, "flops": f}
    if path == "step":
        b, f = _attention_work(case["batch"], 1, case["keys"], case["heads"], case["kv_heads"], case["head_dim"], case["least"])
        return {"bytes": b, "flops": f}
    if path in ("prefill", "decode"):
        hidden, h, hkv, d = QWEN3
        n, t = (h + 2 * hkv) * d, case.get("seq", 1)
        rows = case["batch"] * t
        # x, the residual and the weights in; the sum, the keys, the values and the attention's rows out.
        b = 2 * (3 * rows * hidden + n * hidden + 2 * rows * hkv * d + rows * h * d)
        f = 2 * rows * n * hidden
        if path == "decode":
            cached, g = _attention_work(case["batch"], 1, case["keys"], h, hkv, d, case["least"])
            return {"bytes": b + cached - 4 * rows * h * d, "flops": f + g}
        return {"bytes": b, "flops": f + _attention_work(case["batch"], t, t, h, hkv, d, case["least"], True)[1]}
    if path == "local":
        hidden, h, hkv, d = MODERNBERT
        n, rows = (h + 2 * hkv) * d, case["batch"] * case["seq"]
        f = _attention_work(case["batch"], case["seq"], case["seq"], h, hkv, d, case["least"], False, case["window"])[1]
        return {"bytes": 2 * (rows * hidden + n * hidden + rows * h * d), "flops": 2 * rows * n * hidden + f}
    if path == "prologue":
        _, h, hkv, d = QWEN3
        b, t = case["batch"], case["seq"]
        return {"bytes": 2 * (2 * b * t * (h + 2 * hkv) * d + t * d), "flops": 8 * b * t * (h + hkv) * d}
    if path == "norm":
        tensors = 4 if case["form"].startswith("add_") else 2
        return {"bytes": 2 * (tensors * case["tokens"] + 1) * case["width"], "flops": 6 * case["tokens"] * case["width"]}
    hidden, h, hkv, d = LAYERS[case["layer"]]
    b, t = case["batch"], case["seq"]
    n = (h + 2 * hkv) * d
    return {"bytes": 2 * (b * t * hidden + n * hidden + b * t * n), "flops": 2 * b * t * n * hidden}


def tolerance(case):
    # A norm or a prologue rounds its results once; a contraction's summands and probabilities are 16-bit too.
    once = case["path"] in ("prologue", "norm")
    if case["dtype"] == "f16":
        return {"rel": 1e-3 if once else 2e-3}
    return {"rel": 4e-3 if once else 1e-2}
