"""Performance cases: the work a user of this Provider has it do, through its
public Python entry points (`magnetar_hip.ops`, `magnetar_hip.decoder`).

A case is a dict of plain values. `prepare` makes what a user's program holds
before the call (device inputs, weights, caches, outputs), `run` makes one
pass, `work` states what the pass cannot do without, `tolerance` how far
another correct implementation at the same precision may be, and `exact` is
the same mathematics in 64 bits.

Buffers are torch tensors seen by the library as DeviceArray views, so that
outputs can be looked at without a copy through the host.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "magnetar-provider-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import magnetar_hip  # noqa: E402
from magnetar_hip import ops  # noqa: E402
from magnetar_hip.decoder import WEIGHT_NAMES, DecoderBlock, Shapes  # noqa: E402

_DEVICE = None


def _dev():
    """The program's one bound device."""
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = magnetar_hip.Device(0)
    return _DEVICE


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------

def listed():
    return [
        # A tiny Llama-style block (hidden 256, 4 heads of 64, FFN 688) over a
        # 32-token prompt: the smallest call, where launches and latency count.
        _block("block_tiny_prompt", hidden=256, heads=4, kv_heads=4, ffn=688, vocab=1024, seq=32,
               position=0, compact=False),
        # A 7B-sized block (hidden 4096, 32 heads of 128, FFN 11008) over a
        # prompt of ordinary, odd length, f32 weights.
        _block("block_prompt", hidden=4096, heads=32, kv_heads=32, ffn=11008, vocab=32000, seq=509,
               position=0, compact=False),
        # The same block generating one token against 2048 cached ones.
        _block("block_decode", hidden=4096, heads=32, kv_heads=32, ffn=11008, vocab=32000, seq=1,
               position=2048, compact=False),
        # A grouped-query block with compact bf16 weights (a bf16 checkpoint)
        # generating one token in the middle of a conversation.
        _block("block_decode_compact", hidden=4096, heads=32, kv_heads=8, ffn=14336, vocab=32000,
               seq=1, position=1235, compact=True),
        # The square product on its own, f32.
        _matmul("matmul_square", 4096, 4096, 4096),
        # An FFN projection of a ragged prompt over a compact bf16 weight.
        _matmul("matmul_prompt_compact", 777, 4096, 11008, compact=True),
        # The same projection for a batch of sequences decoding together,
        # added to the residual stream.
        _matmul("matmul_batch_decode", 24, 4096, 11008, addend=2),
        # The output head of one decode step over a tied embedding (weights
        # stored [vocab, hidden]), and the probabilities over the vocabulary.
        {"name": "head_tied", "kind": "head", "m": 1, "hidden": 4096, "vocab": 32000, "tied": True},
        # Causal attention over whole prompts, batched.
        _attention("attention_prompt", batch=4, seq=2048, kv=2048, heads=32, kv_heads=32, d=128),
        # Grouped-query attention of a batch of decode steps.
        _attention("attention_decode", batch=8, seq=1, kv=4096, heads=32, kv_heads=8, d=128),
        # The bandwidth-bound steps of a layer over many tokens: RMSNorm,
        # RoPE, the gated activation and the residual add.
        {"name": "layer_steps", "kind": "steps", "rows": 8192, "heads": 32, "d": 128},
        # The half-precision path on a large odd-sized tensor.
        {"name": "half_add", "kind": "half", "n": 64_000_003, "op": "add", "dtype": "bf16"},
    ]


def _block(name, **kw):
    return dict({"name": name, "kind": "block"}, **kw)


def _matmul(name, m, k, n, ta=False, tb=False, addend=0, compact=False):
    return {"name": name, "kind": "matmul", "m": m, "k": k, "n": n, "ta": ta, "tb": tb,
            "addend": addend, "compact": compact}


def _attention(name, batch, seq, kv, heads, kv_heads, d, causal=True, window=0):
    return {"name": name, "kind": "attention", "batch": batch, "seq": seq, "kv": kv, "heads": heads,
            "kv_heads": kv_heads, "d": d, "causal": causal, "window": window}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MOST_FLOPS, _MOST_BYTES = 1.3e11, 1.0e9  # of a drawn case


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            del case["name"]
            return case


def _draw(rng):
    kind = rng.choice(["block", "block", "matmul", "matmul", "matmul", "head", "attention",
                       "attention", "steps", "half"])
    if kind == "block":
        d = rng.choice([64, 128, 128])
        heads = rng.choice([4, 8, 16, 32])
        group = rng.choice([1, 1, 2, 4])
        return _block("", hidden=heads * d, heads=heads, kv_heads=heads // group,
                      ffn=16 * max(8, int(heads * d * rng.uniform(2.5, 3.6) / 16)),
                      vocab=rng.choice([1024, 32000]),
                      seq=1 if rng.random() < 0.4 else _log_int(rng, 2, 600),
                      position=rng.choice([0, _log_int(rng, 16, 2048)]),
                      compact=rng.random() < 0.4)
    if kind == "matmul":
        m = _log_int(rng, 1, 4096)
        k = rng.choice([256, 688, 1024, 2048, 4096, 4096, 11008, _log_int(rng, 200, 8000)])
        n = rng.choice([256, 1024, 2048, 4096, 4096, 11008, _log_int(rng, 200, 12000)])
        compact = rng.random() < 0.35
        return _matmul("", m, k, n, ta=not compact and rng.random() < 0.1, tb=rng.random() < 0.25,
                       addend=rng.choice([0, 0, 1, 2]), compact=compact)
    if kind == "head":
        return {"name": "", "kind": "head", "m": _log_int(rng, 1, 64),
                "hidden": rng.choice([1024, 2048, 4096]), "vocab": _log_int(rng, 8000, 50000),
                "tied": rng.random() < 0.5}
    if kind == "attention":
        heads = rng.choice([8, 16, 32])
        group = rng.choice([1, 2, 4, 8])
        d = rng.choice([64, 64, 128, 128, 128, 96])
        if rng.random() < 0.5:
            seq, kv = 1, _log_int(rng, 100, 8192)
        else:
            seq = _log_int(rng, 16, 2048)
            kv = seq + rng.choice([0, 0, _log_int(rng, 16, 2048)])
        causal = seq == 1 or rng.random() < 0.85
        window = _log_int(rng, 128, 2048) if causal and rng.random() < 0.25 else 0
        return _attention("", _log_int(rng, 1, 8), seq, kv, heads, heads // group, d, causal, window)
    if kind == "steps":
        return {"name": "", "kind": "steps", "rows": _log_int(rng, 16, 8192),
                "heads": rng.choice([8, 16, 32]), "d": rng.choice([64, 128])}
    return {"name": "", "kind": "half", "n": _log_int(rng, 10_000, 80_000_000),
            "op": rng.choice(["add", "mul"]), "dtype": rng.choice(["f16", "bf16"])}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + 17)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    t = torch.empty(shape, device="cuda").normal_(mean, std, generator=g)
    return t


def _bf16_bits(g, shape, std):
    """A bf16 weight as the bit patterns a checkpoint holds."""
    return _normal(g, shape, std).to(torch.bfloat16).view(torch.int16)


def _widen(bits):
    return bits.view(torch.bfloat16).to(torch.float64)


def _ids(g, n, vocab):
    return torch.randint(0, vocab, (n,), device="cuda", generator=g).to(torch.float32)


def _shapes(c):
    return Shapes(vocab=c["vocab"], hidden=c["hidden"], heads=c["heads"], kv_heads=c["kv_heads"],
                  head_dim=c["hidden"] // c["heads"], ffn=c["ffn"])


def _inputs(c, seed):
    """The case's inputs as torch tensors, from the seed alone."""
    g = _gen(seed)
    kind = c["kind"]
    if kind == "block":
        s = _shapes(c)
        t = {}
        for name, shape in s.weight_shapes().items():
            if name.endswith("norm"):
                t[name] = _normal(g, shape, 0.1, 1.0)
            elif c["compact"]:
                t[name] = _bf16_bits(g, shape, 0.02)
            else:
                t[name] = _normal(g, shape, 0.02)
        kv = s.kv_heads * s.head_dim
        rows = c["position"] + c["seq"]
        for name in ("k_cache", "v_cache"):
            t[name] = _normal(g, (rows, kv), 0.5)
            t[name][c["position"]:] = 0.0
        t["ids"] = _ids(g, c["seq"], c["vocab"])
        return t
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        t = {"a": _normal(g, (k, m) if c["ta"] else (m, k))}
        bshape = (n, k) if c["tb"] else (k, n)
        t["b"] = _bf16_bits(g, bshape, 0.02) if c["compact"] else _normal(g, bshape, 0.02)
        if c["addend"]:
            t["addend"] = _normal(g, (n,) if c["addend"] == 1 else (m, n))
        return t
    if kind == "head":
        h, v = c["hidden"], c["vocab"]
        return {"a": _normal(g, (c["m"], h)), "b": _normal(g, (v, h) if c["tied"] else (h, v), 0.02)}
    if kind == "attention":
        B, H, Hk, d = c["batch"], c["heads"], c["kv_heads"], c["d"]
        return {"q": _normal(g, (B * c["seq"], H * d)), "k": _normal(g, (B * c["kv"], Hk * d)),
                "v": _normal(g, (B * c["kv"], Hk * d))}
    if kind == "steps":
        shape = (c["rows"], c["heads"] * c["d"])
        return {"x": _normal(g, shape), "up": _normal(g, shape), "gain": _normal(g, shape[1:], 0.1, 1.0)}
    dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float16
    return {"a": _normal(g, (c["n"],)).to(dt).view(torch.int16),
            "b": _normal(g, (c["n"],)).to(dt).view(torch.int16)}


def _view(t, half=None):
    """A torch tensor as the library sees it."""
    dtype = np.uint16 if t.dtype == torch.int16 else np.float32
    return magnetar_hip.DeviceArray(_dev(), t.data_ptr(), tuple(t.shape), dtype, half, owned=False)


def _half(c):
    return magnetar_hip.MHIP_BF16 if c["dtype"] == "bf16" else magnetar_hip.MHIP_F16


def prepare(case, seed):
    c, dev = case, _dev()
    t = _inputs(c, seed)
    v = {name: _view(x) for name, x in t.items()}
    st = {"case": c, "t": t, "v": v}
    out = {}
    kind = c["kind"]
    if kind == "block":
        block = DecoderBlock(dev, _shapes(c), {n: v[n] for n in WEIGHT_NAMES},
                             cache_rows=c["position"] + c["seq"], max_seq=c["seq"],
                             bf16_weights=c["compact"])
        block.k_cache, block.v_cache = v["k_cache"], v["v_cache"]
        st["block"] = block
        out["hidden"] = torch.empty((c["seq"], c["hidden"]), device="cuda")
    elif kind == "matmul":
        out["c"] = torch.empty((c["m"], c["n"]), device="cuda")
    elif kind == "head":
        out["logits"] = torch.empty((c["m"], c["vocab"]), device="cuda")
        out["probs"] = torch.empty((c["m"], c["vocab"]), device="cuda")
    elif kind == "attention":
        st["params"] = ops.attention_params(c["seq"], c["kv"], c["heads"], c["d"],
                                            kv_head_count=c["kv_heads"], causal=c["causal"],
                                            window_size=c["window"] or None, batch=c["batch"])
        out["o"] = torch.empty_like(t["q"])
    elif kind == "steps":
        st["rope"] = ops.rope_params(c["d"], c["heads"])
        for name in ("norm", "rotated", "gated", "sum"):
            out[name] = torch.empty_like(t["x"])
    else:
        out["y"] = torch.empty_like(t["a"])
    st["out"] = out
    st["ov"] = {name: _view(x) for name, x in out.items()}
    torch.cuda.synchronize()  # the inputs were made on torch's stream
    return st


def run(state):
    c, v, o, dev = state["case"], state["v"], state["ov"], _dev()
    kind = c["kind"]
    out = state["out"]
    if kind == "block":
        state["block"].forward(v["ids"], c["position"], o["hidden"])
        return {"hidden": out["hidden"], "k_cache": state["t"]["k_cache"],
                "v_cache": state["t"]["v_cache"]}
    if kind == "matmul":
        product = ops.matmul_bf16w if c["compact"] else ops.matmul
        product(dev, v["a"], v["b"], c["ta"], c["tb"], v.get("addend"), c["addend"], o["c"])
        return out["c"]
    if kind == "head":
        ops.matmul(dev, v["a"], v["b"], False, c["tied"], out=o["logits"])
        ops.softmax_rows(dev, o["logits"], o["probs"])
        return out
    if kind == "attention":
        ops.attention(dev, v["q"], v["k"], v["v"], state["params"], o["o"])
        return out["o"]
    if kind == "steps":
        ops.rmsnorm(dev, v["x"], v["gain"], 1e-5, out=o["norm"])
        ops.rope(dev, o["norm"], state["rope"], out=o["rotated"])
        ops.silu_mul(dev, o["norm"], v["up"], out=o["gated"])
        ops.add(dev, v["x"], o["gated"], out=o["sum"])
        return out
    ops.half_binary(dev, v["a"], v["b"], c["op"], _half(c), o["y"])
    return out["y"]


# --------------------------------------------------------------------------
# What a pass cannot do without, and how close its results are
# --------------------------------------------------------------------------

def _admitted(c):
    """(query, key) pairs of one head and batch row."""
    seq, kv, win = c["seq"], c["kv"], c["window"]
    if not c["causal"]:
        return seq * kv
    total = 0
    for i in range(seq):
        keys = kv - seq + i + 1
        total += min(keys, win) if win else keys
    return total


def work(case):
    c = case
    kind = c["kind"]
    if kind == "block":
        h, f, d = c["hidden"], c["ffn"], c["hidden"] // c["heads"]
        kv, s, p = c["kv_heads"] * d, c["seq"], c["position"]
        weights = 2 * h * h + 2 * h * kv + 3 * h * f
        pairs = sum(p + i + 1 for i in range(s))
        size = 2 if c["compact"] else 4
        # weights, the prompt's table rows, cached K/V read, new K/V and output written
        nbytes = size * (weights + s * h) + 4 * (2 * h + 2 * p * kv + 2 * s * kv + s * h + s)
        return {"bytes": nbytes, "flops": 2.0 * s * weights + 4.0 * d * pairs * c["heads"]}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        add = {0: 0, 1: n, 2: m * n}[c["addend"]]
        return {"bytes": 4 * (m * k + m * n + add) + (2 if c["compact"] else 4) * k * n,
                "flops": 2.0 * m * k * n}
    if kind == "head":
        m, h, v = c["m"], c["hidden"], c["vocab"]
        return {"bytes": 4 * (m * h + h * v + 3 * m * v), "flops": 2.0 * m * h * v}
    if kind == "attention":
        d, B = c["d"], c["batch"]
        span = min(c["kv"], c["window"] + c["seq"] - 1) if c["window"] else c["kv"]
        return {"bytes": 4 * B * d * (2 * c["seq"] * c["heads"] + 2 * span * c["kv_heads"]),
                "flops": 4.0 * d * B * c["heads"] * _admitted(c)}
    if kind == "steps":
        n = c["rows"] * c["heads"] * c["d"]
        # four calls: read 1, 1, 2 and 2 tensors, write one each
        return {"bytes": 4 * (10 * n + c["heads"] * c["d"]), "flops": 0}
    return {"bytes": 6 * c["n"], "flops": 0}


def tolerance(case):
    # About four times the 2-norm errors measured against 64 bits: products
    # 1.1e-6 over 4096 terms (2.3e-6 over 16384, 2.5e-7 over 256), the head's
    # probabilities 1.8e-6, attention 4.6e-7, the row steps 9e-8, a block's
    # output 3.2e-6 after a prompt.
    return {"half": "exact", "matmul": {"rel": 6e-6}, "head": {"rel": 8e-6},
            "attention": {"rel": 2e-6}, "steps": {"rel": 5e-7}, "block": {"rel": 1.3e-5}}[case["kind"]]


# --------------------------------------------------------------------------
# 64 bits
# --------------------------------------------------------------------------

def _f64(x):
    return _widen(x) if x.dtype == torch.int16 else x.to(torch.float64)


def _rms(x, gain):
    return x * torch.rsqrt(torch.mean(x * x, -1, keepdim=True) + float(np.float32(1e-5))) * gain


def _rope(x, heads, d, position):
    """Interleaved pairs; the angle is the f32 product of an f32 position and
    an f32 frequency, as the operation is defined."""
    rows = x.shape[0]
    pair = np.arange(d // 2, dtype=np.float32)
    freq = np.power(np.float64(10000.0), (np.float32(-2.0) * pair / np.float32(d)).astype(np.float64))
    freq = torch.from_numpy(freq.astype(np.float32)).cuda()
    pos = torch.arange(position, position + rows, device="cuda").to(torch.float32)
    angle = (pos[:, None] * freq[None, :]).to(torch.float64)[:, None, :]
    y = x.reshape(rows, heads, d // 2, 2)
    a, b = y[..., 0], y[..., 1]
    cos, sin = torch.cos(angle), torch.sin(angle)
    return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).reshape(rows, heads * d)


def _attend(q, k, v, heads, kv_heads, d, causal=True, window=0):
    """One batch row: q [seq, H*d], k and v [kv, Hkv*d]."""
    seq, kv = q.shape[0], k.shape[0]
    scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
    qpos = torch.arange(kv - seq, kv, device="cuda")[:, None]
    keys = torch.arange(kv, device="cuda")[None, :]
    keep = torch.ones((seq, kv), dtype=torch.bool, device="cuda")
    if causal:
        keep &= keys <= qpos
        if window:
            keep &= keys > qpos - window
    out = torch.empty((seq, heads * d), dtype=torch.float64, device="cuda")
    group = heads // kv_heads
    for h in range(heads):
        g = h // group
        kt = k[:, g * d:(g + 1) * d].t().contiguous()
        s = (q[:, h * d:(h + 1) * d].contiguous() @ kt) * scale
        p = torch.softmax(s.masked_fill_(~keep, float("-inf")), -1)
        out[:, h * d:(h + 1) * d] = p @ v[:, g * d:(g + 1) * d].contiguous()
    return out


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "half":
        return None
    t = {name: _f64(x) for name, x in _inputs(c, seed).items()}
    if kind == "block":
        s, pos = _shapes(c), c["position"]
        x = t["embedding"][t["ids"].long()]
        h = _rms(x, t["attn_norm"])
        q = _rope(h @ t["wq"], s.heads, s.head_dim, pos)
        t["k_cache"][pos:] = _rope(h @ t["wk"], s.kv_heads, s.head_dim, pos)
        t["v_cache"][pos:] = h @ t["wv"]
        a = _attend(q, t["k_cache"], t["v_cache"], s.heads, s.kv_heads, s.head_dim)
        x2 = a @ t["wo"] + x
        h2 = _rms(x2, t["ffn_norm"])
        gate = h2 @ t["w_gate"]
        f = gate * torch.sigmoid(gate) * (h2 @ t["w_up"])
        return {"hidden": f @ t["w_down"] + x2, "k_cache": t["k_cache"], "v_cache": t["v_cache"]}
    if kind == "matmul":
        a = t["a"].t().contiguous() if c["ta"] else t["a"]
        b = t["b"].t().contiguous() if c["tb"] else t["b"]
        y = a @ b
        return y + t["addend"] if c["addend"] else y
    if kind == "head":
        logits = t["a"] @ (t["b"].t().contiguous() if c["tied"] else t["b"])
        return {"logits": logits, "probs": torch.softmax(logits, -1)}
    if kind == "attention":
        rows, keys = c["seq"], c["kv"]
        return torch.cat([_attend(t["q"][b * rows:(b + 1) * rows], t["k"][b * keys:(b + 1) * keys],
                                  t["v"][b * keys:(b + 1) * keys], c["heads"], c["kv_heads"], c["d"],
                                  c["causal"], c["window"]) for b in range(c["batch"])])
    norm = _rms(t["x"], t["gain"])
    gated = norm * torch.sigmoid(norm) * t["up"]
    return {"norm": norm, "rotated": _rope(norm, c["heads"], c["d"], 0), "gated": gated,
            "sum": t["x"] + gated}
