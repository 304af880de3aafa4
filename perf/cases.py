"""What the backend's speed is measured on: the calls of a transformer's forward pass
(text and image), from one decoded token to a batch of long prompts, through the
methods of puter_amd.Backend.

Every case holds its device buffers (inputs, weights, outputs, workspaces) as a
program that owns its memory plan does; a pass is the calls alone.  `exact`
computes the same values in float64 with plain torch.
"""
import math

import torch

import puter_amd
from puter_amd import backend as pb

TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
CODE = {"f32": pb.F32, "bf16": pb.BF16, "f16": pb.F16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
PAGE = 16  # tokens per KV page


# ---------------------------------------------------------------- the cases --
def listed():
    return [
        # A pre-norm attention block on a short prompt in f32: eight small calls, so
        # launches and the host's share of them are most of it.
        {"name": "block_f32_128x512", "kind": "block", "dtype": "f32", "seq": 128, "hidden": 512, "heads": 8},
        # One token through one decoder layer, batch 1: what a chat user waits for.
        # Fifteen calls; the weights are read once each.
        {"name": "decode_layer_b1", "kind": "decode_layer", "batch": 1, "ctx": 1000, "hidden": 4096, "heads": 32,
         "kv": 8, "dim": 128, "inter": 14336},
        # The gated MLP over a prompt of 2000 tokens (not a multiple of a tile).
        {"name": "mlp_bf16_2000", "kind": "mlp", "dtype": "bf16", "rows": 2000, "hidden": 4096, "inter": 14336},
        # The output head of a model whose vocabulary is odd: logits for a handful of rows.
        {"name": "head_bf16_33x4096x32001", "kind": "head", "dtype": "bf16", "rows": 33, "hidden": 4096,
         "vocab": 32001},
        # The fused residual + norm between two sub-layers, a long prompt.
        {"name": "gr_rmsnorm_bf16_16384x4096", "kind": "norm", "op": "gr_rms", "dtype": "bf16", "rows": 16384,
         "hidden": 4096, "batches": 1},
        # The modulated norm of an image transformer's block: 4096 latent and 512 text
        # tokens at a hidden size that is not a power of two.
        {"name": "modulated_ln_bf16_4608x3072", "kind": "norm", "op": "modulated", "dtype": "bf16", "rows": 4608,
         "hidden": 3072, "batches": 1},
        # Rotary embedding of Q and K, the gated activation and its widening to f32.
        {"name": "rope_swiglu_cast_8192", "kind": "rope_act", "dtype": "bf16", "rows": 8192, "heads": 32, "kv": 8,
         "dim": 128, "inter": 14336, "mode": 1, "llama3": False},
        # Rotary embedding over text and image axes, the image transformer's queries.
        {"name": "multi_axis_rope_4608", "kind": "axes", "dtype": "bf16", "batch": 1, "side": 64, "text": 512,
         "heads": 24, "dim": 128, "axes": 4},
        # Causal grouped-query prefill of four long prompts.
        {"name": "prefill_bf16_b4_4096", "kind": "attention", "dtype": "bf16", "batch": 4, "seq_q": 4096,
         "seq_k": 4096, "heads": 32, "kv": 8, "dim": 128, "causal": True, "window": 0},
        # The second chunk of a ragged prompt (keys of the first are cached), a head size
        # between the two usual ones.
        {"name": "prefill_f16_700of1500_d96", "kind": "attention", "dtype": "f16", "batch": 2, "seq_q": 700,
         "seq_k": 1500, "heads": 16, "kv": 16, "dim": 96, "causal": True, "window": 0},
        # A decode step's cache traffic for 64 sequences of very different lengths, fp8
        # pages: quantising write of the new rows, then attention over the pages.
        {"name": "paged_fp8_b64", "kind": "paged", "cache": "fp8", "batch": 64, "ctx_lo": 512, "ctx_hi": 8192,
         "heads": 32, "kv": 8},
        # Single-head attention in f32 over a thousand positions and more (a vision encoder's
        # or an autoencoder's mid block calls it head by head).
        {"name": "flash_f32_2048_d64", "kind": "flash", "dtype": "f32", "seq_q": 2048, "seq_k": 2048, "dim": 64,
         "value_dim": 64, "causal": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "decode_layer", "mlp", "head", "norm", "norm", "rope_act", "axes", "attention",
                       "attention", "paged", "flash"])
    if kind == "block":
        heads = rng.choice([4, 8, 12, 16])
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16", "f16"]), "seq": _log(rng, 16, 640),
                "hidden": 64 * heads, "heads": heads}
    if kind == "decode_layer":
        kv, group = rng.choice([(8, 4), (8, 2), (4, 7), (16, 1), (4, 4)])
        hidden = kv * group * 128
        return {"kind": kind, "batch": _log(rng, 1, 64), "ctx": _log(rng, 17, 6000), "hidden": hidden,
                "heads": kv * group, "kv": kv, "dim": 128, "inter": 8 * (hidden * rng.randint(20, 28) // 64)}
    if kind == "mlp":
        hidden = rng.choice([1024, 1536, 2048, 2560, 3072, 4096])
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16"]), "rows": _log(rng, 16, 2000),
                "hidden": hidden, "inter": 8 * (hidden * rng.randint(20, 28) // 64)}
    if kind == "head":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": _log(rng, 1, 256),
                "hidden": rng.choice([768, 1024, 2048, 4096]), "vocab": _log(rng, 8000, 50000)}
    if kind == "norm":
        hidden = rng.choice([8 * _log(rng, 48, 1024), 256 * rng.randint(2, 32), _log(rng, 384, 8192)])
        rows = min(_log(rng, 1, 65536), 16384 * 4096 // hidden)
        batches = rng.choice([1, 1, 2, 4])
        return {"kind": kind, "op": rng.choice(["rms", "ln", "adaptive", "modulated", "gr_rms", "gr_ln"]),
                "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": max(1, rows // batches) * batches,
                "hidden": hidden, "batches": batches}
    if kind == "rope_act":
        kv = rng.choice([2, 4, 8])
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": _log(rng, 1, 4096),
                "heads": kv * rng.choice([1, 2, 4]), "kv": kv, "dim": rng.choice([64, 80, 96, 128]),
                "inter": rng.choice([_log(rng, 1000, 14336), 256 * rng.randint(4, 56)]), "mode": rng.choice([0, 1]),
                "llama3": rng.random() < 0.4}
    if kind == "axes":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "batch": rng.choice([1, 1, 2]),
                "side": rng.randint(12, 64), "text": rng.randint(0, 512), "heads": rng.choice([8, 16, 24]),
                "dim": rng.choice([64, 128]), "axes": rng.choice([3, 4])}
    if kind == "attention":
        dim = rng.choice([64, 64, 80, 96, 128, 128, 256])
        kv, group = rng.choice([(8, 1), (16, 1), (4, 4), (8, 4), (2, 6)])
        seq_k = _log(rng, 40, 3000)
        seq_q = rng.choice([seq_k, seq_k, max(1, seq_k // rng.randint(2, 9)), 1])
        window = rng.choice([0, 0, 0, rng.randint(16, 1024)])
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "batch": rng.choice([1, 2]),
                "seq_q": seq_q, "seq_k": seq_k, "heads": kv * group, "kv": kv, "dim": dim,
                "causal": rng.random() < 0.7, "window": window}
    if kind == "paged":
        lo = _log(rng, 1, 2048)
        return {"kind": kind, "cache": rng.choice(["fp8", "bf16", "f16"]), "batch": _log(rng, 1, 64), "ctx_lo": lo,
                "ctx_hi": min(8192, lo * rng.randint(1, 8)), "heads": rng.choice([8, 32]), "kv": 8}
    dim = rng.choice([40, 64, 64, 80, 128, 256, 512])
    seq = _log(rng, 60, 3000)
    return {"kind": "flash", "dtype": rng.choice(["f32", "f32", "bf16", "f16"]), "seq_q": seq,
            "seq_k": rng.choice([seq, seq, max(1, seq // 3)]), "dim": dim, "value_dim": dim,
            "causal": rng.random() < 0.4}


# ------------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    return torch.randn(shape, device="cuda", generator=g).mul_(std).add_(mean).to(TORCH[dtype])


def _weight(g, rows, cols, dtype):
    return _normal(g, (rows, cols), dtype, 1 / math.sqrt(rows))


def _gamma(g, n, dtype):
    return _normal(g, (n,), dtype, 0.02, 1.0)


def _lengths(c, seed):
    """Context lengths of the sequences, the new token included: evenly spread over the
    range, in the seed's order."""
    n, lo, hi = c["batch"], c["ctx_lo"], c["ctx_hi"]
    g = torch.Generator().manual_seed(seed + 1)
    spread = torch.tensor([lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)], dtype=torch.int32)
    return spread[torch.randperm(n, generator=g)]


def _tables(lengths, seed):
    """A page table over a pool of exactly the pages needed, randomly permuted; the
    last token's page and slot of each sequence."""
    pages = (lengths + PAGE - 1) // PAGE
    total, most = int(pages.sum()), int(pages.max())
    perm = torch.randperm(total, generator=torch.Generator().manual_seed(seed + 2)).to(torch.int32)
    table = torch.zeros((len(lengths), most), dtype=torch.int32)
    at = 0
    for b, n in enumerate(pages.tolist()):
        table[b, :n] = perm[at:at + n]
        at += n
    last = lengths - 1
    ids = table[torch.arange(len(lengths)), (last // PAGE).long()].contiguous()
    return total, table, ids, (last % PAGE).to(torch.int32)


def _inputs(c, seed):
    g, k, t = _gen(seed), c["kind"], {}
    dt = c.get("dtype", "bf16")
    if k == "block":
        s, h = c["seq"], c["hidden"]
        t["x"], t["gamma"] = _normal(g, (s, h), dt), _gamma(g, h, dt)
        t["w"] = [_normal(g, (h, h), dt, 0.02 * math.sqrt(512 / h)) for _ in range(4)]
    elif k == "decode_layer":
        b, h, q, kv, inter = c["batch"], c["hidden"], c["heads"] * c["dim"], c["kv"] * c["dim"], c["inter"]
        lengths = torch.full((b,), c["ctx"], dtype=torch.int32)
        total, table, ids, slots = _tables(lengths, seed)
        t["total"] = total
        t["table"], t["ids"], t["slots"], t["lengths"] = table.cuda(), ids.cuda(), slots.cuda(), lengths.cuda()
        t["x"] = _normal(g, (b, h), dt)
        t["gamma1"], t["gamma2"], t["mod"] = _gamma(g, h, dt), _gamma(g, h, dt), _normal(g, (1, 3 * h), dt)
        t["wq"], t["wk"], t["wv"] = _weight(g, h, q, dt), _weight(g, h, kv, dt), _weight(g, h, kv, dt)
        t["wo"] = _weight(g, q, h, dt)
        t["gate"], t["up"], t["down"] = _weight(g, h, inter, dt), _weight(g, h, inter, dt), _weight(g, inter, h, dt)
        t["kpool"] = _normal(g, (total, PAGE, c["kv"], c["dim"]), dt)
        t["vpool"] = _normal(g, (total, PAGE, c["kv"], c["dim"]), dt)
    elif k == "mlp":
        t["x"] = _normal(g, (c["rows"], c["hidden"]), dt)
        t["gate"], t["up"] = (_weight(g, c["hidden"], c["inter"], dt) for _ in range(2))
        t["down"] = _weight(g, c["inter"], c["hidden"], dt)
    elif k == "head":
        t["x"] = _normal(g, (c["rows"], c["hidden"]), dt)
        t["w"] = _weight(g, c["hidden"], c["vocab"], dt)
    elif k == "norm":
        r, h = c["rows"], c["hidden"]
        t["x"] = _normal(g, (r, h), dt)
        t["branch"] = _normal(g, (r, h), dt) if c["op"].startswith("gr") else None
        t["mod"] = _normal(g, (c["batches"], 6 * h), dt, 0.5)
        t["gamma"], t["beta"] = _gamma(g, h, dt), _normal(g, (h,), dt, 0.02)
    elif k == "rope_act":
        r, d = c["rows"], c["dim"]
        t["q"], t["k"] = _normal(g, (r, c["heads"], d), dt), _normal(g, (r, c["kv"], d), dt)
        t["gate"], t["up"] = _normal(g, (r, c["inter"]), dt), _normal(g, (r, c["inter"]), dt)
    elif k == "axes":
        t["x"] = _normal(g, (c["batch"], c["text"] + c["side"] ** 2, c["heads"], c["dim"]), dt)
    elif k == "attention":
        d, std = c["dim"], c["dim"] ** -0.25  # scores of about one, as after a normalised Q and K
        t["q"] = _normal(g, (c["batch"], c["seq_q"], c["heads"], d), dt, std)
        t["k"] = _normal(g, (c["batch"], c["seq_k"], c["kv"], d), dt, std)
        t["v"] = _normal(g, (c["batch"], c["seq_k"], c["kv"], d), dt)
    elif k == "paged":
        lengths = _lengths(c, seed)
        total, table, ids, slots = _tables(lengths, seed)
        t["total"], t["longest"] = total, int(lengths.max())
        t["table"], t["ids"], t["slots"], t["lengths"] = table.cuda(), ids.cuda(), slots.cuda(), lengths.cuda()
        io, shape = _io(c), (total, PAGE, c["kv"], 128)
        t["q"] = _normal(g, (c["batch"], c["heads"], 128), io)
        t["knew"], t["vnew"] = (_normal(g, (c["batch"], c["kv"], 128), io) for _ in range(2))
        if c["cache"] == "fp8":
            t["kscale"] = torch.rand(c["kv"], device="cuda", generator=g) * 0.002 + 0.01
            t["vscale"] = torch.rand(c["kv"], device="cuda", generator=g) * 0.002 + 0.01
            t["kpool"], t["vpool"] = (_codes(torch.randn(shape, device="cuda", generator=g), t[s])
                                      for s in ("kscale", "vscale"))
        else:
            t["kpool"], t["vpool"] = _normal(g, shape, io), _normal(g, shape, io)
    else:
        t["q"] = _normal(g, (c["seq_q"], c["dim"]), dt)
        t["k"] = _normal(g, (c["seq_k"], c["dim"]), dt)
        t["v"] = _normal(g, (c["seq_k"], c["value_dim"]), dt)
    return t


def _codes(x, scale):
    """x [.., kv, dim] as saturated fp8 codes of x / scale[kv]."""
    return (x / scale.view(-1, 1)).clamp(-448, 448).to(torch.float8_e4m3fn)


def _io(c):
    return "bf16" if c["cache"] == "fp8" else c["cache"]


def _empty(shape, dtype):
    return torch.empty(shape, device="cuda", dtype=TORCH[dtype])


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    dt, k = c.get("dtype", "bf16"), c["kind"]
    if k == "block":
        for n in ("h", "q", "k", "v", "o", "y"):
            t["_" + n] = _empty((c["seq"], c["hidden"]), dt)
    elif k == "decode_layer":
        b = c["batch"]
        for n, w in (("n1", c["hidden"]), ("q", c["heads"] * c["dim"]), ("k", c["kv"] * c["dim"]),
                     ("v", c["kv"] * c["dim"]), ("a", c["heads"] * c["dim"]), ("o", c["hidden"]),
                     ("hid", c["hidden"]), ("n2", c["hidden"]), ("g", c["inter"]), ("u", c["inter"]),
                     ("act", c["inter"]), ("y", c["hidden"])):
            t["_" + n] = _empty((b, w), dt)
    elif k == "mlp":
        for n in ("g", "u", "act"):
            t["_" + n] = _empty((c["rows"], c["inter"]), dt)
        t["_y"] = _empty((c["rows"], c["hidden"]), dt)
    elif k == "head":
        t["_y"] = _empty((c["rows"], c["vocab"]), dt)
    elif k == "norm":
        t["_hid"], t["_y"] = torch.empty_like(t["x"]), torch.empty_like(t["x"])
    elif k == "rope_act":
        t["_q"], t["_k"], t["_act"] = (torch.empty_like(t[n]) for n in ("q", "k", "gate"))
        t["_wide"] = _empty(t["gate"].shape, "f32")
    elif k == "axes":
        t["_y"] = torch.empty_like(t["x"])
    elif k in ("attention", "paged"):
        t["_y"] = torch.empty_like(t["q"])
    else:
        t["_y"] = _empty((c["seq_q"], c["value_dim"]), dt)
    be = puter_amd.Backend()
    if k in ("decode_layer", "paged"):
        t["_longest"] = c["ctx"] if k == "decode_layer" else t["longest"]
        t["_wsb"] = be.PagedDecodeWorkspaceBytes(c["batch"], c["heads"], 128, t["_longest"])
        t["_ws"] = torch.empty(t["_wsb"], device="cuda", dtype=torch.uint8)
    return c, be, t


# -------------------------------------------------------------------- a pass --
def run(state):
    c, be, t = state
    return RUN[c["kind"]](c, be, t, CODE[c.get("dtype", "bf16")])


def _run_block(c, be, t, f):
    s, h, n = c["seq"], c["hidden"], c["heads"]
    be.RMSNorm(pb.RMSNormConfig(1e-6), t["x"], t["gamma"], t["_h"], s, h, f)
    for name, w in (("_q", 0), ("_k", 1), ("_v", 2)):
        be.Matmul(t[name], t["_h"], t["w"][w], s, h, h, f)
    rope = pb.RoPEConfig(BaseFreq=10000.0)
    be.RoPE(rope, t["_q"], t["_q"], s, n, 64, f)
    be.RoPE(rope, t["_k"], t["_k"], s, n, 64, f)
    be.MultiHeadAttention(pb.MultiHeadAttentionConfig(n, 64, True, 0, 0.0, n), t["_q"], t["_k"], t["_v"], t["_o"],
                          s, s, f)
    be.Matmul(t["_y"], t["_o"], t["w"][3], s, h, h, f)
    return t["_y"]


def _run_decode_layer(c, be, t, f):
    b, h, d, inter = c["batch"], c["hidden"], c["dim"], c["inter"]
    q, kv, total = c["heads"] * d, c["kv"] * d, t["total"]
    be.RMSNorm(pb.RMSNormConfig(1e-5), t["x"], t["gamma1"], t["_n1"], b, h, f)
    be.Matmul(t["_q"], t["_n1"], t["wq"], b, h, q, f)
    be.Matmul(t["_k"], t["_n1"], t["wk"], b, h, kv, f)
    be.Matmul(t["_v"], t["_n1"], t["wv"], b, h, kv, f)
    # the sequences stand at one position: a row of batch x heads heads
    rope = pb.RoPEConfig(BaseFreq=500000.0, StartPosition=c["ctx"] - 1, Mode=pb.RoPEModeHalf)
    be.RoPE(rope, t["_q"], t["_q"], 1, b * c["heads"], d, f)
    be.RoPE(rope, t["_k"], t["_k"], 1, b * c["kv"], d, f)
    be.KVPageWrite(t["kpool"], t["_k"], t["ids"], t["slots"], t["kpool"], total, PAGE, kv, b, 0, f)
    be.KVPageWrite(t["vpool"], t["_v"], t["ids"], t["slots"], t["vpool"], total, PAGE, kv, b, 0, f)
    be.PagedDecodeAttention(t["_q"], t["kpool"], t["vpool"], t["table"], t["lengths"], b, t["table"].shape[1], PAGE,
                            total, c["heads"], c["kv"], d, t["_longest"], None, None, f, t["_a"], t["_ws"], t["_wsb"])
    be.Matmul(t["_o"], t["_a"], t["wo"], b, q, h, f)
    be.GatedResidualRMSNorm(pb.RMSNormConfig(1e-5), t["x"], t["_o"], t["mod"], t["gamma2"], t["_hid"], t["_n2"], b,
                            h, b, 3 * h, 0, f)
    _run_ffn(be, t, t["_n2"], b, h, inter, f)
    return t["_hid"], t["_y"], t["kpool"], t["vpool"]


def _run_ffn(be, t, x, rows, h, inter, f):
    be.Matmul(t["_g"], x, t["gate"], rows, h, inter, f)
    be.Matmul(t["_u"], x, t["up"], rows, h, inter, f)
    be.SwiGLUTensors(t["_act"], t["_g"], t["_u"], rows * inter, f)
    be.Matmul(t["_y"], t["_act"], t["down"], rows, inter, h, f)


def _run_mlp(c, be, t, f):
    _run_ffn(be, t, t["x"], c["rows"], c["hidden"], c["inter"], f)
    return t["_y"]


def _run_head(c, be, t, f):
    be.Matmul(t["_y"], t["x"], t["w"], c["rows"], c["hidden"], c["vocab"], f)
    return t["_y"]


def _run_norm(c, be, t, f):
    r, h, op = c["rows"], c["hidden"], c["op"]
    per = r // c["batches"]
    if op == "rms":
        be.RMSNorm(pb.RMSNormConfig(1e-5), t["x"], t["gamma"], t["_y"], r, h, f)
    elif op == "ln":
        be.LayerNorm(t["x"], t["gamma"], t["beta"], t["_y"], r, h, f)
    elif op == "adaptive":
        be.AdaptiveRMSNorm(pb.RMSNormConfig(1e-6), t["x"], t["mod"], t["_y"], r, h, per, 6 * h, f)
    elif op == "modulated":
        be.ModulatedLayerNorm(pb.ModulatedLayerNormConfig(1e-6, 1), t["x"], t["mod"], t["_y"], r, h, per, 6 * h, f)
    elif op == "gr_rms":
        be.GatedResidualRMSNorm(pb.RMSNormConfig(1e-5), t["x"], t["branch"], t["mod"], t["gamma"], t["_hid"],
                                t["_y"], r, h, per, 6 * h, 0, f)
    else:
        be.GatedResidualLayerNorm(t["x"], t["branch"], t["mod"], t["gamma"], t["beta"], t["_hid"], t["_y"], r, h,
                                  per, 6 * h, 0, f)
    return (t["_hid"], t["_y"]) if op.startswith("gr") else t["_y"]


def _rope_config(c):
    if c["llama3"]:
        return pb.RoPEConfig(500000.0, 0, c["mode"], pb.RoPEScalingLlama3, 8.0, 1.0, 4.0, 8192)
    return pb.RoPEConfig(BaseFreq=500000.0, Mode=c["mode"])


def _run_rope_act(c, be, t, f):
    r, n = c["rows"], c["rows"] * c["inter"]
    be.RoPE(_rope_config(c), t["q"], t["_q"], r, c["heads"], c["dim"], f)
    be.RoPE(_rope_config(c), t["k"], t["_k"], r, c["kv"], c["dim"], f)
    be.SwiGLUTensors(t["_act"], t["gate"], t["up"], n, f)
    be.Cast(t["_wide"], pb.F32, t["_act"], f, n)
    return t["_q"], t["_k"], t["_act"], t["_wide"]


def _axis_dims(c):
    d = c["dim"]
    return [d // 4] * 4 if c["axes"] == 4 else [d // 8, 7 * d // 16, 7 * d // 16]


def _run_axes(c, be, t, f):
    cfg = pb.MultiAxisRoPEConfig(10000.0, c["side"] ** 2, c["side"], c["axes"], *_axis_dims(c))
    be.MultiAxisRoPE(cfg, t["x"], t["_y"], c["batch"], t["x"].shape[1], c["heads"], c["dim"], f)
    return t["_y"]


def _run_attention(c, be, t, f):
    cfg = pb.MultiHeadAttentionConfig(c["heads"], c["dim"], c["causal"], c["window"], 0.0, c["kv"])
    be.MultiHeadAttentionBatched(cfg, t["q"], t["k"], t["v"], t["_y"], c["batch"], c["seq_q"], c["seq_k"], f)
    return t["_y"]


def _run_paged(c, be, t, _):
    kv, inner, total, b = c["kv"], c["kv"] * 128, t["total"], c["batch"]
    f = CODE[_io(c)]
    if c["cache"] == "fp8":
        be.KVPageWriteFP8(t["kpool"], t["knew"], t["ids"], t["slots"], total, PAGE, kv, 128, b, 0, t["kscale"], f)
        be.KVPageWriteFP8(t["vpool"], t["vnew"], t["ids"], t["slots"], total, PAGE, kv, 128, b, 0, t["vscale"], f)
    else:
        be.KVPageWrite(t["kpool"], t["knew"], t["ids"], t["slots"], t["kpool"], total, PAGE, inner, b, 0, f)
        be.KVPageWrite(t["vpool"], t["vnew"], t["ids"], t["slots"], t["vpool"], total, PAGE, inner, b, 0, f)
    be.PagedDecodeAttention(t["q"], t["kpool"], t["vpool"], t["table"], t["lengths"], b, t["table"].shape[1], PAGE,
                            total, c["heads"], kv, 128, t["_longest"], t.get("kscale"), t.get("vscale"),
                            pb.F8E4M3 if c["cache"] == "fp8" else f, t["_y"], t["_ws"], t["_wsb"])
    return t["_y"], t["kpool"], t["vpool"]


def _run_flash(c, be, t, f):
    be.FlashAttention(pb.FlashAttentionConfig(64, c["causal"]), t["q"], t["k"], t["v"], t["_y"], c["seq_q"],
                      c["seq_k"], c["dim"], c["value_dim"], f)
    return t["_y"]


RUN = {"block": _run_block, "decode_layer": _run_decode_layer, "mlp": _run_mlp, "head": _run_head,
       "norm": _run_norm, "rope_act": _run_rope_act, "axes": _run_axes, "attention": _run_attention,
       "paged": _run_paged, "flash": _run_flash}


# ------------------------------------------------------------------ the work --
def _pairs(c):
    """(query, key) pairs that the mask lets through, one head of one sequence."""
    sq, sk = c["seq_q"], c["seq_k"]
    causal, window = c["causal"], c.get("window", 0)
    shift = sk - sq if c["kind"] == "attention" else 0
    q = torch.arange(sq, dtype=torch.int64)
    hi = torch.clamp(q + shift + 1, 0, sk) if causal else torch.full_like(q, sk)
    lo = torch.clamp(q - window + 1, min=0) if window else torch.zeros_like(q)
    return int(torch.clamp(hi - lo, min=0).sum())


def work(case):
    c, k = case, case["kind"]
    e = SIZE[c.get("dtype", "bf16")]
    if k == "block":
        s, h = c["seq"], c["hidden"]
        return {"bytes": e * (4 * h * h + 2 * s * h), "flops": 8 * s * h * h + 2 * s * (s + 1) * h}
    if k == "decode_layer":
        b, h, q, kv = c["batch"], c["hidden"], c["heads"] * c["dim"], c["kv"] * c["dim"]
        w = 2 * h * q + 2 * h * kv + 3 * h * c["inter"]
        return {"bytes": 2 * (w + 2 * b * c["ctx"] * kv + 3 * b * h), "flops": 2 * b * w + 4 * b * c["ctx"] * q}
    if k == "mlp":
        r, h, i = c["rows"], c["hidden"], c["inter"]
        return {"bytes": e * (3 * h * i + 2 * r * h), "flops": 6 * r * h * i}
    if k == "head":
        r, h, v = c["rows"], c["hidden"], c["vocab"]
        return {"bytes": e * (h * v + r * h + r * v), "flops": 2 * r * h * v}
    if k == "norm":
        n = c["rows"] * c["hidden"]
        return {"bytes": e * n * (4 if c["op"].startswith("gr") else 2), "flops": 8 * n}
    if k == "rope_act":
        n, m = c["rows"] * (c["heads"] + c["kv"]) * c["dim"], c["rows"] * c["inter"]
        return {"bytes": e * (2 * n + 3 * m) + 4 * m, "flops": 3 * n + 8 * m}
    if k == "axes":
        n = c["batch"] * (c["text"] + c["side"] ** 2) * c["heads"] * c["dim"]
        return {"bytes": 2 * e * n, "flops": 3 * n}
    if k == "attention":
        n = c["batch"] * c["dim"]
        return {"bytes": e * n * (2 * c["seq_q"] * c["heads"] + 2 * c["seq_k"] * c["kv"]),
                "flops": 4 * n * c["heads"] * _pairs(c)}
    if k == "paged":
        tokens = c["batch"] * (c["ctx_lo"] + c["ctx_hi"]) // 2
        size = 1 if c["cache"] == "fp8" else 2
        return {"bytes": 2 * size * tokens * c["kv"] * 128 + 4 * c["batch"] * (c["heads"] + c["kv"]) * 128,
                "flops": 4 * tokens * c["heads"] * 128}
    n = c["seq_q"] * (c["dim"] + c["value_dim"]) + c["seq_k"] * (c["dim"] + c["value_dim"])
    return {"bytes": e * n, "flops": 2 * (c["dim"] + c["value_dim"]) * _pairs(c)}


def tolerance(case):
    k, dt = case["kind"], case.get("dtype", "bf16")
    return {"rel": TOLERANCE[_io(case) if k == "paged" else dt][k]}


# about four times the largest relative error against float64 that was measured over
# seeded draws of each kind: the rounding of the stored values and the order of the sums
# (a chain of calls adds up its own; the activations' and flash attention's exponential
# is the reference's polynomial, good to a few 1e-5)
TOLERANCE = {
    "f32": {"block": 2e-6, "head": 3e-6, "norm": 1e-6, "rope_act": 2.5e-5, "axes": 1e-6, "attention": 2e-6,
            "flash": 1e-4},
    "bf16": {"block": 1.4e-2, "decode_layer": 2e-2, "mlp": 1.4e-2, "head": 7e-3, "norm": 8e-3, "rope_act": 7e-3,
             "axes": 6e-3, "attention": 8e-3, "paged": 1.2e-2, "flash": 1.2e-2},
    "f16": {"block": 2e-3, "mlp": 2e-3, "head": 1e-3, "norm": 1e-3, "rope_act": 1e-3, "axes": 1e-3,
            "attention": 1e-3, "paged": 2e-3, "flash": 2.4e-3},
}


# ------------------------------------------------------------------- float64 --
def exact(case, seed):
    c, t = case, _inputs(case, seed)
    return EXACT[c["kind"]](c, {n: _wide(n, v) for n, v in t.items()})


def _wide(name, v):
    if isinstance(v, list):
        return [x.double() for x in v]
    keep = not isinstance(v, torch.Tensor) or v.dtype == torch.int32
    return v if keep else v.double()


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _ln(x, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps)


def _rotate(x, angle, half):
    """x [rows, heads, dim] rotated by angle [rows, dim / 2]."""
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    n = x.shape[-1] // 2
    a, b = (x[..., :n], x[..., n:]) if half else (x[..., 0::2], x[..., 1::2])
    a, b = a * cos - b * sin, a * sin + b * cos
    return torch.cat((a, b), -1) if half else torch.stack((a, b), -1).flatten(-2)


def _angles(positions, dim, base):
    inv = base ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float64) / dim)
    return torch.as_tensor(positions, device="cuda", dtype=torch.float64)[:, None] * inv


def _softmax_product(q, k, v, causal, window, shift):
    """One head: q [sq, d], k [sk, d], v [sk, dv]."""
    s = q @ k.t().contiguous() / math.sqrt(q.shape[-1])
    qi = torch.arange(q.shape[0], device="cuda")[:, None]
    ki = torch.arange(k.shape[0], device="cuda")[None]
    if causal:
        s.masked_fill_(ki > qi + shift, -math.inf)
    if window:
        s.masked_fill_(qi - ki >= window, -math.inf)
    return torch.nan_to_num(torch.softmax(s, -1)) @ v


def _heads(q, k, v, causal, window, shift):
    """q [sq, heads, d], k and v [sk, kv, d]."""
    group = q.shape[1] // k.shape[1]
    out = [_softmax_product(q[:, h].contiguous(), k[:, h // group].contiguous(), v[:, h // group].contiguous(),
                            causal, window, shift) for h in range(q.shape[1])]
    return torch.stack(out, 1)


def _exact_block(c, t):
    s, n = c["seq"], c["heads"]
    h = _rms(t["x"], 1e-6) * t["gamma"]
    q, k, v = ((h @ w).view(s, n, 64) for w in t["w"][:3])
    a = _angles(range(s), 64, 10000.0)
    o = _heads(_rotate(q, a, False), _rotate(k, a, False), v, True, 0, 0)
    return o.reshape(s, -1) @ t["w"][3]


def _paged_heads(c, t, q, kpool, vpool):
    """q [batch, heads, d] over the pages of each sequence."""
    out = []
    for b, n in enumerate(t["lengths"].tolist()):
        pages = t["table"][b, :(n + PAGE - 1) // PAGE].long()
        k, v = (p[pages].flatten(0, 1)[:n] for p in (kpool, vpool))
        out.append(_heads(q[b:b + 1], k, v, False, 0, 0)[0])
    return torch.stack(out)


def _write(c, t, pool, rows):
    pool = pool.clone()
    pool[t["ids"].long(), t["slots"].long()] = rows
    return pool


def _exact_decode_layer(c, t):
    b, d = c["batch"], c["dim"]
    n1 = _rms(t["x"], 1e-5) * t["gamma1"]
    a = _angles([c["ctx"] - 1] * b, d, 500000.0)
    q = _rotate((n1 @ t["wq"]).view(b, -1, d), a, True)
    k = _rotate((n1 @ t["wk"]).view(b, -1, d), a, True)
    kpool, vpool = _write(c, t, t["kpool"], k), _write(c, t, t["vpool"], (n1 @ t["wv"]).view(b, -1, d))
    att = _paged_heads(c, t, q, kpool, vpool).reshape(b, -1)
    hid = t["x"] + t["mod"][0, 2 * c["hidden"]:] * (att @ t["wo"])
    return hid, _exact_mlp(c, {**t, "x": _rms(hid, 1e-5) * t["gamma2"]}), kpool, vpool


def _exact_mlp(c, t):
    return (torch.nn.functional.silu(t["x"] @ t["gate"]) * (t["x"] @ t["up"])) @ t["down"]


def _exact_norm(c, t):
    h, op, x = c["hidden"], c["op"], t["x"]
    mod = t["mod"].repeat_interleave(c["rows"] // c["batches"], 0)
    if op == "adaptive":
        return _rms(x, 1e-6) * (1 + mod[:, :h]) + mod[:, h:2 * h]
    if op == "modulated":
        return _ln(x, 1e-6) * (1 + mod[:, 4 * h:5 * h]) + mod[:, 3 * h:4 * h]
    if op.startswith("gr"):
        x = x + mod[:, 2 * h:3 * h] * t["branch"]
    y = _rms(x, 1e-5) * t["gamma"] if op.endswith("rms") else _ln(x, 1e-5) * t["gamma"] + t["beta"]
    return (x, y) if op.startswith("gr") else y


def _exact_rope_act(c, t):
    a = _angles(range(c["rows"]), c["dim"], 500000.0)
    if c["llama3"]:
        inv = a.new_tensor(500000.0) ** (-torch.arange(0, c["dim"], 2, device="cuda").double() / c["dim"])
        wave = 2 * math.pi / inv
        smooth = (8192 / wave - 1.0) / (4.0 - 1.0)
        mixed = (1 - smooth) * inv / 8.0 + smooth * inv
        inv = torch.where(wave > 8192 / 1.0, inv / 8.0, torch.where(wave < 8192 / 4.0, inv, mixed))
        a = torch.arange(c["rows"], device="cuda").double()[:, None] * inv
    act = torch.nn.functional.silu(t["gate"]) * t["up"]
    return _rotate(t["q"], a, c["mode"] == 1), _rotate(t["k"], a, c["mode"] == 1), act, act


def _exact_axes(c, t):
    """Text tokens stand at their index on the text axis (the last of four, the first of
    fewer) and at 0 on the others; image tokens at their row on axis 1, column on axis 2."""
    seq, text = t["x"].shape[1], c["text"]
    i = torch.arange(seq, device="cuda", dtype=torch.float64)
    image = i >= text
    row, col = torch.div(i - text, c["side"], rounding_mode="floor"), torch.remainder(i - text, c["side"])
    zero, angles = torch.zeros_like(i), []
    for axis, d in enumerate(_axis_dims(c)):
        pos = torch.where(image, row if axis == 1 else col if axis == 2 else zero,
                          i if axis == (3 if c["axes"] == 4 else 0) else zero)
        angles.append(_angles(pos, d, 10000.0))
    a = torch.cat(angles, 1)
    return torch.stack([_rotate(x, a, False) for x in t["x"]])


def _exact_attention(c, t):
    return torch.stack([_heads(q, k, v, c["causal"], c["window"], c["seq_k"] - c["seq_q"])
                        for q, k, v in zip(t["q"], t["k"], t["v"])])


def _exact_paged(c, t):
    knew, vnew, kpool, vpool = t["knew"], t["vnew"], t["kpool"], t["vpool"]
    if c["cache"] == "fp8":  # the pools hold codes: the new rows are rounded to them here too
        ks, vs = t["kscale"].view(-1, 1), t["vscale"].view(-1, 1)
        knew, vnew = (_codes(n.float(), s.float()).double() for n, s in ((knew, ks), (vnew, vs)))
        kpool, vpool = _write(c, t, kpool, knew), _write(c, t, vpool, vnew)
        return _paged_heads(c, t, t["q"], kpool * ks, vpool * vs), kpool, vpool
    kpool, vpool = _write(c, t, kpool, knew), _write(c, t, vpool, vnew)
    return _paged_heads(c, t, t["q"], kpool, vpool), kpool, vpool


def _exact_flash(c, t):
    return _softmax_product(t["q"], t["k"], t["v"], c["causal"], 0, 0)


EXACT = {"block": _exact_block, "decode_layer": _exact_decode_layer, "mlp": lambda c, t: _exact_mlp(c, t),
         "head": lambda c, t: t["x"] @ t["w"], "norm": _exact_norm, "rope_act": _exact_rope_act,
         "axes": _exact_axes, "attention": _exact_attention, "paged": _exact_paged, "flash": _exact_flash}
