"""The work that users of this framework have it do, as cases to be timed.

Every case goes through the public entry points (`DecoderModel`, `KvCache`,
the device greedy loop, `pick`) on seeded synthetic weights. The shapes are
the repository's own: the tiny f32 decoder (2 layers, hidden 256), slices of
one to four layers of the 1B shape (hidden 2048, 32 / 8 heads of 64, ffn
8192) and of the 8B shape (hidden 4096, 32 / 8 heads of 128, ffn 14336), the
1B shape whole, and a routed stack (8 experts, top 2). A slice is as deep as
its outputs need to depend on every row of its inputs; its vocabulary is
short, so that the layers are what it measures.

Kinds of pass:
  greedy  a whole request: a prompt, then tokens from the device loop
  prompt  prompts evaluated into an empty cache (prefill)
  step    tokens added to warm caches: one row per sequence (decode), short
          blocks (forced spans), and with "pick" a masked, sampled choice
A "step" state keeps several groups of sequences with the same context and
serves them in turn, so that the context stays near the stated length.
"""
from __future__ import annotations

import json
import math
import struct

import numpy as np
import torch

from esp_amd import DecoderModel, Sampler
from esp_amd.config import DecoderConfig
from esp_amd.model import LoraAdapter
from esp_amd.streaming import ArtifactSource, StreamingOptions

# hidden, heads, kv heads, ffn, RoPE theta
SHAPES = {
    "tiny": (256, 4, 4, 688, 10000.0),
    "1b": (2048, 32, 8, 8192, 500000.0),
    "8b": (4096, 32, 8, 14336, 500000.0),
    "moe": (2048, 32, 8, 7168, 1000000.0),
}
EXPERTS, TOPK = 8, 2
LORA_ALPHA = 32.0
EPS = 1e-5
STD = 0.02
ROOM = 384  # positions a step state's sequences can grow by before they are evaluated anew


def _case(kind, shape, layers, fmt, vocab, **kw):
    c = {"kind": kind, "shape": shape, "layers": layers, "format": fmt, "vocab": vocab,
         "kv": "f32", "lora": 0, "seqs": 1, "ctx": 0, "rows": 1, "new": 0, "pick": False}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest use: the tiny f32 decoder answers a short prompt; every launch counts
        _case("greedy", "tiny", 2, "f32", 1024, name="request_tiny_f32", rows=32, new=32),
        # the default f32 format evaluating a chat turn
        _case("prompt", "1b", 2, "f32", 4096, name="prompt_1b_f32", rows=301),
        # one user's request on the whole 1B-shape model, as a chat host runs it
        _case("greedy", "1b", 16, "bf16", 128256, name="request_1b_bf16", rows=512, new=64),
        # one token at a long context with an adapter on q and v: latency per token of one layer
        _case("step", "8b", 1, "bf16", 4096, name="step_8b_lora", ctx=4096, lora=16),
        # a long prompt: the matrix-bound end of the range
        _case("prompt", "8b", 2, "bf16", 4096, name="prompt_8b_bf16", rows=2048),
        # several users' prompts of unequal length in one pass, half-precision cache
        _case("prompt", "1b", 2, "bf16", 4096, name="prompts_1b_bf16", seqs=12, rows=283, kv="f16"),
        # a handful of users decoding together
        _case("step", "8b", 2, "bf16", 4096, name="few_8b_bf16", seqs=4, ctx=700),
        # a loaded server: 64 sequences, some of them forced 8-token spans, masks and sampling
        _case("step", "1b", 4, "bf16", 32000, name="serve_1b_bf16", seqs=64, ctx=1024, rows=8, pick=True),
        # a grammar's forced span on a 4-bit model
        _case("step", "8b", 2, "q4-block32", 4096, name="span_8b_q4", ctx=500, rows=9),
        # a document-sized prompt on an 8-bit model
        _case("prompt", "8b", 2, "q8-block32", 4096, name="prompt_8b_q8", rows=1100),
        # a few users decoding together on a routed model: every expert's rows are few
        _case("step", "moe", 2, "bf16", 4096, name="few_moe_bf16", seqs=6, ctx=300),
        # a prompt on a routed model: grouped expert products over ragged row counts
        _case("prompt", "moe", 2, "bf16", 4096, name="prompt_moe_bf16", rows=777),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("greedy", "prompt", "prompt", "step", "step", "serve"))
    if kind == "greedy":
        return _case("greedy", "tiny", 2, "f32", 1024, rows=_log(rng, 2, 512), new=_log(rng, 2, 64))
    if kind == "serve":
        return _case("step", "1b", 2, "bf16", 32000, seqs=rng.randint(16, 64), ctx=_log(rng, 64, 1024),
                     rows=rng.randint(1, 12), pick=True, kv=rng.choice(("f32", "f16")))
    shape, fmt = rng.choice((("1b", "f32"), ("1b", "bf16"), ("8b", "bf16"), ("8b", "q8-block32"),
                             ("1b", "q4-block32"), ("moe", "bf16")))
    kv = rng.choice(("f32", "f16")) if fmt == "bf16" else "f32"
    if kind == "prompt":
        seqs = rng.choice((1, 1, 1, 5))
        return _case("prompt", shape, 2, fmt, 4096, seqs=seqs, kv=kv,
                     rows=_log(rng, 2, (1024 if fmt == "f32" else 2048) // seqs))
    lora = 16 if (shape, fmt) == ("1b", "bf16") and rng.random() < 0.5 else 0
    most = (8, 512) if fmt == "f32" else (24, 2048)
    return _case("step", shape, 2, fmt, 4096, seqs=_log(rng, 1, most[0]), ctx=_log(rng, 16, most[1]),
                 kv=kv, lora=lora, rows=rng.choice((1, 1, 1, _log(rng, 2, 24))))


# ------------------------------------------------------------------ geometry

def _config(c):
    H, nq, nkv, F, theta = SHAPES[c["shape"]]
    max_pos = 8192
    if c["shape"] == "moe":
        return DecoderConfig.mixtral_style(
            vocab_size=c["vocab"], hidden_size=H, intermediate_size=F, num_hidden_layers=c["layers"],
            num_attention_heads=nq, num_key_value_heads=nkv, max_position_embeddings=max_pos,
            rms_norm_eps=EPS, rope_theta=theta, num_experts=EXPERTS, num_experts_per_tok=TOPK,
            moe_intermediate_size=F)
    raw = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": H,
           "intermediate_size": F, "num_hidden_layers": c["layers"], "num_attention_heads": nq,
           "num_key_value_heads": nkv, "max_position_embeddings": max_pos, "rms_norm_eps": EPS,
           "rope_theta": theta, "vocab_size": c["vocab"], "tie_word_embeddings": _tied(c),
           "hidden_act": "silu"}
    return DecoderConfig.from_json_bytes(json.dumps(raw).encode())


def _tied(c):
    return c["shape"] == "1b" and not c["format"].startswith("q")


def _synthetic(c):
    """The whole 1B-shape model takes the library's own seeded weights (2.5 GB
    of artifacts would be most of a preparation); slices are loaded."""
    return c["kind"] == "greedy" and c["shape"] == "1b"


def _block_lens(c):
    """Tokens that each sequence of one pass brings."""
    n, B = c["rows"], c["seqs"]
    if c["pick"]:  # every eighth sequence is inside a forced span, the others decode
        return [n if i % 8 == 0 else 1 for i in range(B)]
    if c["kind"] == "prompt" and B > 1:  # ragged
        return [max(1, n * (7 * i % B + 1) // B) for i in range(B)]
    return [n] * B


def _ids(rng, n, vocab):
    return rng.integers(0, vocab, n).astype(np.int32)


def _inputs(c, seed):
    """Token ids: each sequence's context, then the block it brings."""
    rng = np.random.default_rng([seed, 1])
    groups = _groups(c)
    ctx = [[_ids(rng, c["ctx"], c["vocab"]) for _ in range(c["seqs"])] for _ in range(groups)]
    blocks = [_ids(rng, n, c["vocab"]) for n in _block_lens(c)]
    return ctx, blocks


def _groups(c):
    if c["kind"] != "step":
        return 1
    return 8 if c["seqs"] == 1 else 4 if c["seqs"] <= 24 else 2


# ------------------------------------------------------------------- weights

def _normal(gen, shape, std):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std)


def _quantize(w, bits):
    """Block-32 symmetric integers along the rows and their f32 scales."""
    top = 127.0 if bits == 8 else 7.0
    b = w.view(w.shape[0], -1, 32)
    scale = (b.abs().amax(2) / top).clamp_min(1e-30)
    q = torch.round(b / scale[:, :, None]).clamp_(-top, top).to(torch.int8)
    return q.view(w.shape), scale


def _weights(c, seed):
    """(name, kind, tensors) of every weight, made on the GPU from the seed:
    kind "proj" in the case's format, "vec" f32 or f16, "embed"."""
    H, nq, nkv, F, _ = SHAPES[c["shape"]]
    hd = H // nq
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + 17)
    fmt = c["format"]

    def proj(name, rows, cols):
        w = _normal(gen, (rows, cols), STD)
        if fmt == "f32":
            return name, "proj", (w,)
        if fmt == "bf16":
            return name, "proj", (w.to(torch.bfloat16),)
        return name, "packed", _quantize(w, 8 if fmt.startswith("q8") else 4)

    def vec(name, n):
        w = 1.0 + _normal(gen, (n,), 0.1)
        return name, "vec", (w.to(torch.float16 if fmt.startswith("q") else torch.float32),)

    e = _normal(gen, (c["vocab"], H), STD)
    edt = torch.float32 if fmt == "f32" else torch.bfloat16 if fmt == "bf16" else torch.float16
    yield "model.embed_tokens.weight", "embed", (e.to(edt),)
    yield vec("model.norm.weight", H)
    if not _tied(c):
        yield proj("lm_head.weight", c["vocab"], H)
    for l in range(c["layers"]):
        p = "model.layers.%d." % l
        yield vec(p + "input_layernorm.weight", H)
        yield vec(p + "post_attention_layernorm.weight", H)
        yield proj(p + "self_attn.q_proj.weight", nq * hd, H)
        yield proj(p + "self_attn.k_proj.weight", nkv * hd, H)
        yield proj(p + "self_attn.v_proj.weight", nkv * hd, H)
        yield proj(p + "self_attn.o_proj.weight", H, nq * hd)
        if c["shape"] == "moe":
            # qwen2_moe layers carry q/k/v biases
            for n, k in (("q", nq * hd), ("k", nkv * hd), ("v", nkv * hd)):
                yield p + "self_attn.%s_proj.bias" % n, "vec", (_normal(gen, (k,), STD),)
            yield proj(p + "mlp.gate.weight", EXPERTS, H)
            for x in range(EXPERTS):
                q = p + "mlp.experts.%d." % x
                yield proj(q + "gate_proj.weight", F, H)
                yield proj(q + "up_proj.weight", F, H)
                yield proj(q + "down_proj.weight", H, F)
        else:
            yield proj(p + "mlp.gate_proj.weight", F, H)
            yield proj(p + "mlp.up_proj.weight", F, H)
            yield proj(p + "mlp.down_proj.weight", H, F)


def _lora_weights(c, seed):
    """A and B of q_proj and v_proj, as f32 values exact in bf16."""
    H, nq, nkv, _, _ = SHAPES[c["shape"]]
    hd = H // nq
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 1000003 + 18)
    out = {}
    for l in range(c["layers"]):
        for m, n in (("q_proj", nq * hd), ("v_proj", nkv * hd)):
            out[l, m] = (_normal(gen, (c["lora"], H), 0.02).to(torch.bfloat16),
                         _normal(gen, (n, c["lora"]), 0.01).to(torch.bfloat16))
    return out


_DTYPE = {torch.float32: "F32", torch.bfloat16: "BF16", torch.float16: "F16"}


def _entry(name, kind, tensors):
    """(name, dtype, shape, byte tensors) as a checkpoint stores it."""
    if kind == "packed":
        q, scale = tensors
        v = q.view(torch.uint8).reshape(-1)
        if int(q.abs().max()) <= 7:  # two 4-bit values a byte, the even input low
            n = (v & 15).view(-1, 2)
            v = n[:, 0] | (n[:, 1] << 4)
        parts = [v, scale.reshape(-1).view(torch.uint8)]
        return name, "U8", [sum(x.numel() for x in parts)], parts
    t = tensors[0].contiguous()
    return name, _DTYPE[t.dtype], list(t.shape), [t.reshape(-1).view(torch.uint8)]


def _artifact(entries):
    """One safetensors file of the entries, in host memory."""
    align = {"F32": 4, "BF16": 2, "F16": 2, "U8": 1}
    header, off, order = {}, 0, sorted(entries, key=lambda e: (-align[e[1]], e[0]))
    for name, dt, shape, parts in order:
        n = sum(x.numel() for x in parts)
        header[name] = {"dtype": dt, "shape": shape, "data_offsets": [off, off + n]}
        off += n
    text = json.dumps(header, separators=(",", ":")).encode()
    text += b" " * (-len(text) % 8)
    head = struct.pack("<Q", len(text)) + text
    host = torch.empty(len(head) + off, dtype=torch.uint8, pin_memory=True)
    host[:len(head)] = torch.frombuffer(bytearray(head), dtype=torch.uint8)
    at = len(head)
    for _, _, _, parts in order:
        for x in parts:
            host[at:at + x.numel()].copy_(x, non_blocking=True)
            at += x.numel()
    torch.cuda.synchronize()
    return host.numpy()


def _model(c, seed):
    cfg = _config(c)
    if _synthetic(c):
        return DecoderModel.synthetic(cfg, seed=seed, std=STD, fmt=c["format"])
    if c["lora"]:  # adapters come with a checkpoint loaded whole
        blob = _artifact([_entry(*w) for w in _weights(c, seed)])
        ad = {}
        for (l, m), (a, b) in _lora_weights(c, seed).items():
            p = "base_model.model.model.layers.%d.self_attn.%s." % (l, m)
            ad[p + "lora_A.weight"], ad[p + "lora_B.weight"] = a, b
        adapter = LoraAdapter(c["lora"], LORA_ALPHA, ["q_proj", "v_proj"],
                              _artifact([_entry(k, "proj", (v,)) for k, v in ad.items()]).tobytes())
        return DecoderModel.from_bytes(cfg, memoryview(blob), c["format"], [adapter])
    shared, layers, experts = [], [[] for _ in range(c["layers"])], {}
    for name, kind, t in _weights(c, seed):
        part = name.split(".")
        if part[1] != "layers":
            shared.append(_entry(name, kind, t))
        elif "experts" in part:
            experts.setdefault((int(part[2]), int(part[5])), []).append(_entry(name, kind, t))
        else:
            layers[int(part[2])].append(_entry(name, kind, t))
    layers = [_artifact(x) for x in layers]
    experts = {k: _artifact(v) for k, v in experts.items()}
    shared = _artifact(shared).tobytes()
    most = max(len(x) for x in layers + list(experts.values()))
    return DecoderModel.from_layer_source(cfg, shared, ArtifactSource(layers, experts),
                                          StreamingOptions(max_layer_bytes=most, max_shared_bytes=len(shared)),
                                          c["format"]).with_resident_layers()


# ---------------------------------------------------------------- the passes

class _Rows:
    """A cache's device buffer of f32 rows, for torch to look at in place. The
    tensor made of it keeps this object, and so the cache whose memory it is."""

    def __init__(self, kv, address, shape):
        self.kv = kv
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (address, False),
                                         "version": 3}


def _device_logits(kv, vocab):
    address, rows = kv.logits_device()
    return torch.as_tensor(_Rows(kv, address, (rows, vocab)), device="cuda")


def _warm(s):
    """Every sequence's context evaluated into the empty cache."""
    s["kv"].reset()
    flat = [x for g in s["ctx"] for x in g]
    for at in range(0, len(flat), 32):
        part = flat[at:at + 32]
        s["model"].forward_batch(s["kv"], range(at, at + len(part)), part, want_logits=False)


def prepare(case, seed):
    c = case
    model = _model(c, seed)
    ctx, blocks = _inputs(c, seed)
    s = {"case": c, "model": model, "ctx": ctx, "blocks": blocks, "turn": 0}
    if c["kind"] == "greedy":
        s["kv"] = model.new_cache(1, c["rows"] + c["new"])
    elif c["kind"] == "prompt":
        s["kv"] = model.new_cache(c["seqs"], max(len(b) for b in blocks), c["kv"])
    else:
        s["kv"] = model.new_cache(c["seqs"] * len(ctx), c["ctx"] + ROOM, c["kv"])
        _warm(s)
    if c["pick"]:
        rng = np.random.default_rng([seed, 2])
        words = (c["vocab"] + 31) // 32
        allow = rng.random((c["seqs"], words * 32), dtype=np.float32) < 0.05
        allow[:, c["vocab"]:] = False
        allow[np.arange(c["seqs"]), rng.integers(0, c["vocab"], c["seqs"])] = True
        s["masks"] = np.packbits(allow, axis=1, bitorder="little").view(np.uint32).copy()
        s["samplers"] = [Sampler(0.8, 0.9, int(seed) * 64 + i) for i in range(c["seqs"])]
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    c, model, kv = s["case"], s["model"], s["kv"]
    if c["kind"] == "greedy":
        kv.reset(0)
        ids = model.generate_greedy_device(kv, s["blocks"][0], c["new"], eos=[])
        return {"ids": np.array(ids), "logits": _device_logits(kv, c["vocab"])}
    if c["kind"] == "prompt":
        kv.reset()
        if c["seqs"] == 1:
            return model.try_forward_cached_last(s["blocks"][0], kv)
        return model.forward_batch(kv, range(c["seqs"]), s["blocks"])
    first = s["turn"] % len(s["ctx"]) * c["seqs"]
    s["turn"] += 1
    seqs = range(first, first + c["seqs"])
    if kv.position(first) + c["rows"] > kv.max_ctx:
        _warm(s)
    if c["pick"]:
        model.forward_batch(kv, seqs, s["blocks"], want_logits=False)
        ids, _ = model.pick(kv, c["seqs"], s["masks"], s["samplers"])
        return {"ids": ids.astype(np.int64), "logits": _device_logits(kv, c["vocab"])}
    if c["seqs"] == 1:
        return model.try_forward_cached_last(s["blocks"][0], kv, first)
    return model.forward_batch(kv, seqs, s["blocks"])


# ------------------------------------------------------------- what it costs

def _layer_weights(c, rows):
    """(bytes, multiply-adds per row) of one layer's projections; a routed
    layer reads the experts that `rows` uniformly routed tokens touch."""
    H, nq, nkv, F, _ = SHAPES[c["shape"]]
    hd = H // nq
    attn = H * (nq + 2 * nkv) * hd + H * nq * hd
    per = {"f32": 4.0, "bf16": 2.0, "q8-block32": 1.125, "q4-block32": 0.625}[c["format"]]
    lora = c["lora"] * (2 * H + (nq + nkv) * hd)
    if c["shape"] != "moe":
        return (attn + 3 * H * F + lora) * per, attn + 3 * H * F + lora
    touched = EXPERTS * (1.0 - (1.0 - TOPK / EXPERTS) ** rows)
    return (attn + EXPERTS * H + touched * 3 * H * F) * per, attn + EXPERTS * H + TOPK * 3 * H * F


def _forward_work(c, ctx, lens):
    H, nq, nkv, _, _ = SHAPES[c["shape"]]
    hd = H // nq
    rows = sum(lens)
    wb, wm = _layer_weights(c, rows)
    per = {"f32": 4.0, "bf16": 2.0, "q8-block32": 1.125, "q4-block32": 0.625}[c["format"]]
    kvb = 2 * nkv * hd * (2 if c["kv"] == "f16" else 4)
    pairs = sum(n * ctx + n * (n + 1) / 2 for n in lens)  # (row, key) pairs
    keys = sum(ctx + 2 * n for n in lens)  # keys read once, new ones written once
    b = c["layers"] * (wb + kvb * keys) + c["vocab"] * H * per + rows * H * 4 + len(lens) * c["vocab"] * 4
    f = c["layers"] * (2.0 * wm * rows + 4.0 * nq * hd * pairs) + 2.0 * len(lens) * c["vocab"] * H
    return b, f


def work(case):
    c = case
    if c["kind"] == "greedy":
        b, f = _forward_work(c, 0, [c["rows"]])
        for i in range(c["new"] - 1):
            b1, f1 = _forward_work(c, c["rows"] + i, [1])
            b, f = b + b1, f + f1
        return {"bytes": b, "flops": f}
    b, f = _forward_work(c, c["ctx"], _block_lens(c))
    if c["pick"]:
        b += c["seqs"] * (c["vocab"] * 4 + c["vocab"] / 8)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the distance from 64 bits that the paths show: f32
    products and sums reach 1e-5, activations split into two bf16 halves with
    32-bit sums 3e-5, a half-precision cache 5e-4. Ids are whole: equal unless
    two scores tie."""
    c = case
    rel = 4e-5 if c["format"] == "f32" else 2e-3 if c["kv"] == "f16" else 1.2e-4
    return {"rel": rel, "max": 10 * rel, "differ": 0.0}


# ------------------------------------------------------------------- 64 bits

def _dense(kind, t):
    if kind == "packed":
        q, scale = t
        return (q.view(q.shape[0], -1, 32).double() * scale.double()[:, :, None]).view(q.shape)
    return t[0].double()


def _rope(c, n):
    """cos and sin of the f32 angles that the model's definition rounds to."""
    H, nq, _, _, theta = SHAPES[c["shape"]]
    hd = H // nq
    e = (np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)).astype(np.float64)
    inv = np.float32(1.0) / np.power(np.float64(np.float32(theta)), e).astype(np.float32)
    ang = (np.arange(n, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float64)
    t = torch.from_numpy(np.concatenate([ang, ang], 1)).cuda()
    return torch.cos(t), torch.sin(t)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _attend(q, k, v, nq, nkv):
    """Causal attention of one sequence, a kv head at a time, in row blocks."""
    S, hd = q.shape[0], q.shape[1] // nq
    G = nq // nkv
    out = torch.empty_like(q)
    pos = torch.arange(S, device=q.device)
    for h in range(nkv):
        kh, vh = k[:, h * hd:(h + 1) * hd], v[:, h * hd:(h + 1) * hd]
        for g in range(h * G, (h + 1) * G):
            sc = q[:, g * hd:(g + 1) * hd] @ kh.t().contiguous() / math.sqrt(hd)
            sc.masked_fill_(pos[None, :] > pos[:, None], float("-inf"))
            out[:, g * hd:(g + 1) * hd] = torch.softmax(sc, 1) @ vh
    return out


def _last_rows(c, seed, seqs):
    """Logits of the last position of each token sequence, in 64 bits."""
    H, nq, nkv, F, _ = SHAPES[c["shape"]]
    hd = H // nq
    ends = np.cumsum([len(s) for s in seqs])
    ids = torch.from_numpy(np.concatenate(seqs).astype(np.int64)).cuda()
    cos, sin = _rope(c, max(len(s) for s in seqs))
    at = torch.cat([torch.arange(len(s), device="cuda") for s in seqs])
    cos, sin = cos[at][:, None, :], sin[at][:, None, :]
    top, weights, lora = {}, _weights(c, seed), _lora_weights(c, seed) if c["lora"] else {}

    def turned(x, heads):
        x = x.view(-1, heads, hd)
        r = torch.cat([-x[..., hd // 2:], x[..., :hd // 2]], -1)
        return (x * cos + r * sin).reshape(-1, heads * hd)

    def take(layer):
        got = {}
        need = 9 if c["shape"] != "moe" else 0
        for name, kind, t in weights:
            if layer is None:
                top[name] = _dense(kind, t)
                if len(top) == (2 if _tied(c) else 3):
                    return top
                continue
            got[name.split(".", 3)[3]] = t if "experts" in name else _dense(kind, t)
            if len(got) == (need or 10 + 3 * EXPERTS):
                return got

    take(None)
    x = top["model.embed_tokens.weight"][ids]
    for l in range(c["layers"]):
        w = take(l)
        n = _norm(x, w["input_layernorm.weight"])
        q, k, v = (n @ w["self_attn.%s_proj.weight" % j].t() for j in "qkv")
        if c["shape"] == "moe":
            q, k, v = (y + w["self_attn.%s_proj.bias" % j] for y, j in zip((q, k, v), "qkv"))
        for m, (a, b) in ((m, t) for (ll, m), t in lora.items() if ll == l):
            d = (LORA_ALPHA / c["lora"]) * (n @ a.double().t()) @ b.double().t()
            q, v = (q + d, v) if m == "q_proj" else (q, v + d)
        q, k = turned(q, nq), turned(k, nkv)
        a = torch.cat([_attend(q[e - len(s):e], k[e - len(s):e], v[e - len(s):e], nq, nkv)
                       for e, s in zip(ends, seqs)])
        x = x + a @ w["self_attn.o_proj.weight"].t()
        n = _norm(x, w["post_attention_layernorm.weight"])
        if c["shape"] != "moe":
            g = torch.nn.functional.silu(n @ w["mlp.gate_proj.weight"].t())
            x = x + (g * (n @ w["mlp.up_proj.weight"].t())) @ w["mlp.down_proj.weight"].t()
            continue
        p = torch.softmax(n @ w["mlp.gate.weight"].t(), 1)
        best, who = torch.topk(p, TOPK, 1)
        best = best / best.sum(1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(EXPERTS):
            rows, slot = (who == e).nonzero(as_tuple=True)
            if len(rows):
                gate, up, down = (_dense("proj", w["mlp.experts.%d.%s_proj.weight" % (e, j)])
                                  for j in ("gate", "up", "down"))
                m = n[rows]
                m = (torch.nn.functional.silu(m @ gate.t()) * (m @ up.t())) @ down.t()
                y[rows] += best[rows, slot, None] * m
        x = x + y
    last = torch.from_numpy(ends - 1).cuda()
    head = top["model.embed_tokens.weight"] if _tied(c) else top["lm_head.weight"]
    return _norm(x[last], top["model.norm.weight"]) @ head.t()


def exact(case, seed):
    c = case
    if _synthetic(c):
        return None  # the library's own weights are not known outside it
    ctx, blocks = _inputs(c, seed)
    if c["kind"] == "greedy":
        seq, ids = [int(t) for t in blocks[0]], []
        for _ in range(c["new"]):
            logits = _last_rows(c, seed, [np.array(seq)])
            ids.append(int(logits[0].argmax()))
            if len(ids) < c["new"]:
                seq.append(ids[-1])
        return {"ids": None, "logits": logits}
    seqs = [np.concatenate([a, b]) for a, b in zip(ctx[0], blocks)]
    logits = _last_rows(c, seed, seqs)
    if c["pick"]:
        return {"ids": None, "logits": logits}
    return logits[0] if c["seqs"] == 1 else logits
