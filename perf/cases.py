"""The workloads whose speed is tracked: one pass each through the public
entry points of the library's Python binding, at the shapes of the Qwen3 and
Qwen3.5 models the library serves.

Seven kinds of work, which `draw` spreads over their whole range of sizes:

  chain      the five layer ops between a layer's contractions (RMSNorm, q/k
             norm + RoPE, add + RMSNorm, SwiGLU, residual add), op by op or in
             one launch, from one decoded token to a long prompt
  mlp        a layer's MLP block on the fp16 projections (norm, gate|up with
             SwiGLU, down with the residual add), from one row to a prompt
  attention  a layer's decode attention over per-sequence KV rings: fused with
             the q/k norm and RoPE as the decode step runs it, or plain
  deltanet   a Qwen3.5 linear-attention layer's decode step
  sample     penalties, softmax and the categorical draw over logits rows
  decode     a whole Qwen3-0.6B decode step with context in every ring
  convert    the bf16 -> fp16 convert of a checkpoint's tensors
"""
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ane-lm_amd"))

import anelm  # noqa: E402

D = 128            # Qwen3's head_dim
THETA = 1e6
EPS = 1e-6
VOCAB = 151936
ROPE_ROWS = 16384
REP, FREQ, WINDOW = 1.2, 0.1, 256   # the sampler's default penalties and window

# hidden, q heads, kv heads, intermediate
MODELS = {"0.6b": (1024, 16, 8, 3072), "4b": (2560, 32, 8, 9728), "8b": (4096, 32, 8, 12288)}
LAYERS_06B = 28
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # a decoded token's layer ops at the smallest model: launches and host calls are what they cost
        dict(name="chain decode 0.6b", kind="chain", model="0.6b", T=1, prefill=False, gamma="bf16", one_launch=False),
        # the layer ops of a long prompt at the largest model: streaming at HBM rate
        dict(name="chain prefill 8b", kind="chain", model="8b", T=8192, prefill=True, gamma="f16", one_launch=False),
        # a small batch's MLP block: bound by reading the weights once
        dict(name="mlp 8 rows 4b", kind="mlp", rows=8, H=2560, I=9728, tiled=False),
        # a prompt's MLP block: bound by the matrix cores
        dict(name="mlp prompt 8b", kind="mlp", rows=2048, H=4096, I=12288, tiled=True),
        # one conversation with a long history
        dict(name="attention one 8b", kind="attention", fused=True, B=1, nq=32, nk=8, dim=128, cap=2048, fill="long"),
        # a serving batch whose conversations have every length up to the ring's capacity
        dict(name="attention ragged 8b", kind="attention", fused=True, B=48, nq=32, nk=8, dim=128, cap=2048, fill="ragged"),
        # a serving batch through a Qwen3.5-0.8B linear-attention layer
        dict(name="deltanet 64", kind="deltanet", B=64, nkh=16, nvh=16, gamma="f32"),
        # sampling for one conversation, and for a serving batch
        dict(name="sample 1", kind="sample", rows=1, vocab=VOCAB, temperature=0.6, ragged=False),
        dict(name="sample 64", kind="sample", rows=64, vocab=VOCAB, temperature=0.6, ragged=True),
        # the whole decode step for one conversation, and for a serving batch
        dict(name="decode one 0.6b", kind="decode", B=1, context=512),
        dict(name="decode batch 0.6b", kind="decode", B=48, context=256),
        # converting the layers of a checkpoint after loading it
        dict(name="convert 0.6b", kind="convert", model="0.6b", layers=28, odd=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("chain", "mlp", "attention", "deltanet", "sample", "decode", "convert"))
    if kind == "chain":
        T = _log(rng, 1, 8192)
        return dict(kind=kind, model=rng.choice(list(MODELS)), T=T, prefill=T > 64 or rng.random() < 0.3,
                    gamma=rng.choice(list(DTYPES)), one_launch=rng.random() < 0.4)
    if kind == "mlp":
        H, I = rng.choice(((1024, 3072), (2560, 9728), (4096, 12288), (2048, 6144), (896, 4864)))
        return dict(kind=kind, rows=_log(rng, 1, 2048), H=H, I=I, tiled=rng.random() < 0.7)
    if kind == "attention":
        fused = rng.random() < 0.6
        dim = 128 if fused else rng.choice((64, 128, 256))
        nk = rng.choice((2, 4, 8))
        return dict(kind=kind, fused=fused, B=_log(rng, 1, 64), nq=nk * rng.choice((1, 2, 4)), nk=nk, dim=dim,
                    cap=_log(rng, 64, 2048 if dim == 256 else 4096), fill=rng.choice(("long", "ragged")))
    if kind == "deltanet":
        nkh = rng.choice((8, 16))
        return dict(kind=kind, B=_log(rng, 1, 64), nkh=nkh, nvh=nkh * rng.choice((1, 1, 2)), gamma=rng.choice(("f32", "bf16")))
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 64), vocab=rng.choice((VOCAB, VOCAB, _log(rng, 8000, VOCAB))),
                    temperature=rng.choice((0.6, 0.6, 1.0, 0.0)), ragged=rng.random() < 0.7)
    if kind == "decode":
        return dict(kind=kind, B=_log(rng, 1, 64), context=_log(rng, 32, 256))
    return dict(kind=kind, model=rng.choice(("0.6b", "4b")), layers=rng.randint(1, 14), odd=rng.choice((0, 0, 1, 3)))


# ------------------------------------------------------------------- inputs

def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * salt + seed)


class _Rand:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = _gen(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda")
        return t if std == 1.0 and mean == 0.0 else t.mul_(std).add_(mean)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo)

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def gamma(self, n, dtype):
        return self.normal(n, std=0.05, mean=1.0).to(DTYPES[dtype])


def _chain_inputs(c, seed):
    H, nq, nk, I = MODELS[c["model"]]
    T, r = c["T"], _Rand(seed)
    s = dict(x=r.normal(T, H), attn=r.normal(T, H), mlp=r.normal(T, H), q=r.normal(T, nq * D), k=r.normal(T, nk * D),
             g=r.normal(T, I), u=r.normal(T, I), w_in=r.gamma(H, c["gamma"]), w_post=r.gamma(H, c["gamma"]),
             wq=r.gamma(D, c["gamma"]), wk=r.gamma(D, c["gamma"]))
    s["pos"] = torch.arange(T, device="cuda", dtype=torch.int32) if c["prefill"] else r.ints(0, 4096, (T,))
    return s


def _mlp_inputs(c, seed):
    r = _Rand(seed)
    return dict(x=r.normal(c["rows"], c["H"]), w=r.gamma(c["H"], "bf16"),
                gu=r.normal(2 * c["I"], c["H"], std=0.02).half(), down=r.normal(c["H"], c["I"], std=0.02).half())


def _lengths(c, r):
    """Rows in each ring: every length up to the capacity once over, in an order of the seed's; or all nearly full."""
    B, cap = c["B"], c["cap"]
    lens = [max(1, round(cap * (i + 0.5) / B)) if c["fill"] == "ragged" else cap - cap // 16 for i in range(B)]
    return torch.tensor(lens, device="cuda", dtype=torch.int32)[torch.randperm(B, generator=r.g, device="cuda")]


def _attention_inputs(c, seed):
    B, nq, nk, dim, cap, r = c["B"], c["nq"], c["nk"], c["dim"], c["cap"], _Rand(seed)
    s = dict(kc=r.normal(B, cap, nk * dim), vc=r.normal(B, cap, nk * dim), qkv=r.normal(B, (nq + 2 * nk) * dim),
             len=_lengths(c, r), start=r.ints(0, cap, (B,)))
    if c["fused"]:
        s.update(wq=r.gamma(D, "bf16"), wk=r.gamma(D, "bf16"), pos=s["len"] - 1)
    return s


def _deltanet_inputs(c, seed):
    B, nkh, nvh, r = c["B"], c["nkh"], c["nvh"], _Rand(seed)
    ch = (2 * nkh + nvh) * D
    s = dict(S=r.normal(B, nvh, D, D, std=0.05), conv=r.normal(B, ch, 3), cw=r.normal(ch, 4, std=0.5), x=r.normal(B, ch),
             z=r.normal(B, nvh * D), decay=r.uniform(B, nvh, lo=0.8), beta=r.uniform(B, nvh), nw=r.gamma(D, c["gamma"]))
    s["pos"] = r.ints(0, 3, (B,))
    return s


def _sample_inputs(c, seed):
    rows, vocab, r = c["rows"], c["vocab"], _Rand(seed)
    s = dict(logits=r.normal(rows, vocab, std=3.0), hist=r.ints(0, vocab, (rows, WINDOW)), r=r.uniform(rows))
    s["hist_len"] = r.ints(0, WINDOW + 1, (rows,)) if c["ragged"] else torch.full((rows,), WINDOW, device="cuda", dtype=torch.int32)
    return s


def _decode_tokens(c, seed):
    """Token ids [context + 1, B]: the context, then the step's."""
    return _Rand(seed).ints(0, VOCAB, (c["context"] + 1, c["B"]))


def _tensors_06b():
    H, nq, nk, I = MODELS["0.6b"]
    t = {"model.embed_tokens.weight": (VOCAB, H), "model.norm.weight": (H,)}
    for i in range(LAYERS_06B):
        t.update({"model.layers.%d.%s.weight" % (i, n): shape for n, shape in (
            ("self_attn.q_proj", (nq * D, H)), ("self_attn.k_proj", (nk * D, H)), ("self_attn.v_proj", (nk * D, H)),
            ("self_attn.o_proj", (H, nq * D)), ("self_attn.q_norm", (D,)), ("self_attn.k_norm", (D,)),
            ("mlp.gate_proj", (I, H)), ("mlp.up_proj", (I, H)), ("mlp.down_proj", (H, I)),
            ("input_layernorm", (H,)), ("post_attention_layernorm", (H,)))})
    return t


def _weights_06b():
    """The tensors of a random checkpoint of Qwen3-0.6B's shapes (bf16), one after the other, always the same."""
    g = _gen(11, 5)
    for name, shape in _tensors_06b().items():
        t = torch.randn(*shape, generator=g, device="cuda")
        yield name, (t.mul_(0.02) if len(shape) > 1 else t.mul_(0.05).add_(1.0)).bfloat16()


def _checkpoint_06b():
    """That checkpoint as a safetensors file, written once."""
    path = os.path.join(tempfile.gettempdir(), "qwen3-0.6b-random-%d.safetensors" % os.getuid())
    head, at = {}, 0
    for name, shape in _tensors_06b().items():
        n = 2 * math.prod(shape)
        head[name] = {"dtype": "BF16", "shape": list(shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    if not os.path.exists(path) or os.path.getsize(path) != 8 + len(text) + at:
        part = "%s.%d" % (path, os.getpid())
        with open(part, "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for _, t in _weights_06b():
                f.write(t.view(torch.int16).cpu().numpy().tobytes())
        os.replace(part, path)
    return path


def _convert_sizes(c):
    H, nq, nk, I = MODELS[c["model"]]
    layer = [H * nq * D, H * nk * D, H * nk * D, H * nq * D, I * H, I * H, H * I, H, H, D, D]
    return [n + c["odd"] for _ in range(c["layers"]) for n in layer]


# ------------------------------------------------------- what a program keeps

def _rope():
    cos, sin = torch.empty(ROPE_ROWS, D // 2, device="cuda"), torch.empty(ROPE_ROWS, D // 2, device="cuda")
    anelm.rope_table(cos, sin, THETA)
    return cos, sin


def _bytes(n):
    return torch.zeros(max(int(n), 16), dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind == "chain":
        s.update(_chain_inputs(c, seed))
        s["cos"], s["sin"] = _rope()
        s.update(xn=torch.empty_like(s["x"]), xp=torch.empty_like(s["x"]), h=torch.empty_like(s["g"]))
    elif kind == "mlp":
        i = _mlp_inputs(c, seed)
        rows, H, I = c["rows"], c["H"], c["I"]
        padded = -(-rows // 16) * 16   # whole 16-row tiles
        s.update(x=i["x"], w=i["w"], a=torch.zeros(padded, H, dtype=torch.float16, device="cuda"),
                 h=torch.zeros(padded, I, dtype=torch.float16, device="cuda"))
        if rows > 16 and c["tiled"]:
            for name, w in (("gu", i["gu"]), ("down", i["down"])):
                s[name] = _bytes(anelm.proj_tiled_size(*w.shape))
                anelm.proj_tile_f16(s[name], w)
        else:
            s.update(gu=i["gu"], down=i["down"])
    elif kind == "attention":
        s.update(_attention_inputs(c, seed))
        B, nq, nk, dim = c["B"], c["nq"], c["nk"], c["dim"]
        s["ws"] = _bytes(anelm.gqa_workspace_size(B, nq, nk, dim, c["cap"]))
        s["out"] = torch.empty(B, nq * dim, device="cuda", dtype=torch.float16 if c["fused"] else torch.float32)
        s["q"], s["k"], s["v"] = s["qkv"].split([nq * dim, nk * dim, nk * dim], dim=1)
        if c["fused"]:
            s["cos"], s["sin"] = _rope()
    elif kind == "deltanet":
        s.update(_deltanet_inputs(c, seed))
        B, nkh, nvh = c["B"], c["nkh"], c["nvh"]
        s["out"] = torch.empty_like(s["z"])
        if nkh == nvh:   # the one-launch step keeps a ring position per head
            s["pos"] = s["pos"].repeat_interleave(nvh).view(B, nvh).contiguous()
        else:
            s["mixed"] = torch.empty_like(s["x"])
            s["q"], s["k"], s["v"] = s["mixed"].split([nkh * D, nkh * D, nvh * D], dim=1)
    elif kind == "sample":
        s.update(_sample_inputs(c, seed))
        s["ids"] = torch.zeros(c["rows"], dtype=torch.int32, device="cuda")
        s["probs"] = torch.zeros_like(s["logits"])
        s["params"] = anelm.SamplingParams(c["temperature"], REP, WINDOW, FREQ)
        s["ws"] = _bytes(anelm.sample_workspace_size(c["rows"], c["vocab"]))
    elif kind == "decode":
        H, nq, nk, I = MODELS["0.6b"]
        B, n = c["B"], c["context"]
        cfg = anelm.Qwen3Config(H, LAYERS_06B, nq, nk, D, I, VOCAB, THETA, EPS)
        s["model"] = anelm.Qwen3Model(_checkpoint_06b(), cfg, max_batch=B, kv_capacity=n)
        s["logits"] = torch.empty(B, VOCAB, device="cuda")
        ids = _decode_tokens(c, seed)
        for t in range(n):   # the conversation so far, token by token; it fills the rings
            s["model"].forward(ids[t], torch.full((B,), t, dtype=torch.int32, device="cuda"), s["logits"])
        s["ids"], s["pos"] = ids[n], torch.full((B,), n, dtype=torch.int32, device="cuda")
    else:
        sizes = _convert_sizes(c)
        src = _Rand(seed).normal(sum(sizes), std=0.02).bfloat16().view(torch.int16)
        s["flat"] = torch.empty_like(src)
        s["src"], s["dst"] = list(src.split(sizes)), list(s["flat"].split(sizes))
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "chain":
        if c["one_launch"]:
            anelm.layer_ops(s["x"], s["xn"], s["xp"], s["attn"], s["mlp"], s["q"], s["k"], s["h"], s["g"], s["u"], s["w_in"],
                            s["w_post"], s["wq"], s["wk"], s["pos"], s["cos"], s["sin"], THETA, EPS)
        else:
            anelm.rmsnorm(s["xn"], s["x"], s["w_in"], EPS)
            anelm.qknorm_rope(s["q"], s["k"], s["wq"], s["wk"], s["pos"], s["cos"], s["sin"], THETA, EPS)
            anelm.add_rmsnorm(s["x"], s["attn"], s["xp"], s["w_post"], EPS)
            anelm.silu_mul(s["h"], s["g"], s["u"])
            anelm.residual_add(s["x"], s["mlp"])
        return [s["x"], s["xn"], s["xp"], s["q"], s["k"], s["h"]]
    if kind == "mlp":
        rows, H, I = c["rows"], c["H"], c["I"]
        if rows <= 16:
            anelm.proj_f16_fused(s["h"][:rows], s["x"], s["gu"], norm=s["w"], eps=EPS, epilogue=anelm.PROJ_SWIGLU_F16)
            anelm.proj_f16_x16_fused(s["x"], s["h"][:rows], s["down"], epilogue=anelm.PROJ_ADD)
        elif c["tiled"]:
            anelm.rmsnorm_f16_tiled(s["a"], s["x"], s["w"], EPS)
            anelm.proj_f16_tt(s["h"], s["a"], s["gu"], rows, I, H, epilogue=anelm.PROJ_SWIGLU_F16_TILED)
            anelm.proj_f16_tt(s["x"], s["h"], s["down"], rows, H, I, epilogue=anelm.PROJ_ADD)
        else:
            anelm.rmsnorm_f16(s["a"][:rows], s["x"], s["w"], EPS)
            anelm.proj_f16_x16_fused(s["h"][:rows], s["a"][:rows], s["gu"], epilogue=anelm.PROJ_SWIGLU_F16)
            anelm.proj_f16_x16_fused(s["x"], s["h"][:rows], s["down"], epilogue=anelm.PROJ_ADD)
        return [s["x"]]
    if kind == "attention":
        if c["fused"]:
            anelm.gqa_attention_qk(s["out"], s["q"], s["k"], s["v"], s["wq"], s["wk"], s["pos"], s["cos"], s["sin"], s["kc"],
                                   s["vc"], s["start"], s["len"], c["nq"], c["nk"], s["ws"], THETA, EPS)
            return [s["out"], s["kc"], s["vc"]]
        anelm.gqa_attention(s["out"], s["q"], s["kc"], s["vc"], s["start"], s["len"], c["nq"], c["nk"], c["dim"], s["ws"])
        return [s["out"]]
    if kind == "deltanet":
        if c["nkh"] == c["nvh"]:
            anelm.conv_ssm_step_gated_norm(s["out"], s["S"], s["conv"], s["pos"], s["x"], s["cw"], s["decay"], s["beta"],
                                           s["z"], s["nw"], D ** -0.5, EPS)
        else:
            anelm.conv1d_silu_l2norm(s["mixed"], s["conv"], s["pos"], s["x"], s["cw"], c["nkh"], D ** -0.5)
            anelm.ssm_step_gated_norm(s["out"], s["S"], s["q"], s["k"], s["v"], s["decay"], s["beta"], s["z"], s["nw"],
                                      c["nkh"], EPS)
        return [s["out"], s["S"], s["conv"], s["pos"]]
    if kind == "sample":
        anelm.sample(s["ids"], s["probs"], s["logits"], s["hist"], s["hist_len"], s["params"], s["r"], s["ws"])
        return [s["ids"]] if c["temperature"] <= 0 else [s["ids"], s["probs"]]
    if kind == "decode":
        s["model"].forward(s["ids"], s["pos"], s["logits"])
        return [s["logits"]]
    anelm.bf16_to_f16_multi(s["dst"], s["src"])
    return [s["flat"].view(torch.float16)]


# -------------------------------------------------------------- what it needs

def work(case):
    c, kind = case, case["kind"]
    if kind == "chain":
        H, nq, nk, I = MODELS[c["model"]]
        T, g = c["T"], 4 if c["gamma"] == "f32" else 2
        # x, attn, mlp in, x and both norms out; q, k in place; cos, sin rows; g, u in, h out; the gammas
        return dict(bytes=4 * T * (6 * H + 2 * (nq + nk) * D + D + 3 * I) + g * (2 * H + 2 * D), flops=T * (12 * H + 10 * (nq + nk) * D + 6 * I))
    if kind == "mlp":
        rows, H, I = c["rows"], c["H"], c["I"]
        return dict(bytes=6 * H * I + 8 * rows * H + 2 * H, flops=6 * rows * H * I)
    if kind == "attention":
        B, nq, nk, dim, cap = c["B"], c["nq"], c["nk"], c["dim"], c["cap"]
        rows = sum(max(1, round(cap * (i + 0.5) / B)) for i in range(B)) if c["fill"] == "ragged" else B * (cap - cap // 16)
        return dict(bytes=8 * rows * nk * dim + B * dim * (4 * (nq + 2 * nk) + (2 if c["fused"] else 4) * nq), flops=4 * rows * nq * dim)
    if kind == "deltanet":
        B, nkh, nvh = c["B"], c["nkh"], c["nvh"]
        ch = (2 * nkh + nvh) * D
        # the states in and out; conv taps, input, one tap out; z, out; the conv weights
        return dict(bytes=4 * (2 * B * nvh * D * D + B * ch * 5 + 2 * B * nvh * D + 4 * ch), flops=8 * B * nvh * D * D)
    if kind == "sample":
        n = c["rows"] * c["vocab"]
        return dict(bytes=4 * n * (1 if c["temperature"] <= 0 else 2) + 4 * c["rows"] * WINDOW, flops=n * (2 if c["temperature"] <= 0 else 30))
    if kind == "decode":
        H, nq, nk, I = MODELS["0.6b"]
        weights = LAYERS_06B * (H * (2 * nq + 2 * nk) * D + 3 * H * I) + VOCAB * H
        rows = LAYERS_06B * c["B"] * c["context"]
        return dict(bytes=2 * weights + 8 * rows * nk * D + 4 * c["B"] * VOCAB, flops=2 * c["B"] * weights + 4 * rows * nq * D)
    n = sum(_convert_sizes(c))
    return dict(bytes=4 * n, flops=0)


def tolerance(case):
    """About four times what the path differs by between its kernels for few and for many rows, whose sums run in
    another order, or, where it has one order, from 64 bits.  fp16 results whose 32-bit sums differ in the last bits
    round to the other neighbour now and then: one unit in the last place of the largest is the "max" there."""
    kind = case["kind"]
    if kind == "convert":
        return "exact"
    if kind == "sample":
        return {"rel": 1.8e-6, "differ": 0.0}   # 2.5e-7 to 4.4e-7 from 64 bits
    if kind == "mlp":
        return {"rel": 4e-4, "max": 0.013}      # 2 to 16 rows against 17: up to 1.0e-4, max 3.1e-3
    if kind == "attention" and case["fused"]:
        return {"rel": 1e-4, "max": 0.02}       # 32-bit outputs 1.7e-7 from 64 bits, then rounded to fp16
    if kind == "decode":
        return {"rel": 4e-3, "max": 0.02}       # 1, 4 and 17 sequences against each other: 1.0e-3, max 4.6e-3
    return {"rel": 1e-6}                        # 32-bit sums: 0.4e-7 to 1.7e-7 from 64 bits


# -------------------------------------------------------------- in 64 bits

def _rms(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _silu(x):
    return x / (1 + torch.exp(-x))


def _rotate(x, pos):
    """Half-split RoPE of x [..., T, heads, D]; pos [T].  The angle is a 32-bit product, as the models define it."""
    e = np.arange(0, D, 2, dtype=np.float32) / np.float32(D)
    inv = np.float32(1) / np.power(np.float64(THETA), e.astype(np.float64)).astype(np.float32)
    a = (pos.to(torch.float32)[:, None] * torch.from_numpy(inv).to(pos.device)[None]).double()
    cos, sin = torch.cos(a)[:, None], torch.sin(a)[:, None]
    lo, hi = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], dim=-1)


def _to_f16_down(x):
    """x (64 bits, within fp16's range) rounded towards zero to fp16's values: ten bits of the significand, or multiples of 2^-24."""
    return torch.where(x.abs() < 2.0 ** -14, (x * 2.0 ** 24).trunc() * 2.0 ** -24, (x.view(torch.int64) >> 42 << 42).view(torch.float64))


def exact(case, seed):
    return {"chain": _exact_chain, "mlp": _exact_mlp, "attention": _exact_attention, "deltanet": _exact_deltanet,
            "sample": _exact_sample, "decode": _exact_decode, "convert": _exact_convert}[case["kind"]](case, seed)


def _exact_chain(c, seed):
    H, nq, nk, I = MODELS[c["model"]]
    i, T = _chain_inputs(c, seed), c["T"]
    x, pos = i["x"].double(), i["pos"]
    xn = _rms(x, i["w_in"])
    q = _rotate(_rms(i["q"].double().view(T, nq, D), i["wq"]), pos).reshape(T, -1)
    k = _rotate(_rms(i["k"].double().view(T, nk, D), i["wk"]), pos).reshape(T, -1)
    x = x + i["attn"].double()
    return [x + i["mlp"].double(), xn, _rms(x, i["w_post"]), q, k, _silu(i["g"].double()) * i["u"].double()]


def _exact_mlp(c, seed):
    i, I = _mlp_inputs(c, seed), c["I"]
    x = i["x"].double()
    a = _rms(x, i["w"])
    g, u = (a @ i["gu"][j * I:(j + 1) * I].double().t().contiguous() for j in (0, 1))
    return [x + (_silu(g) * u) @ i["down"].double().t().contiguous()]


def _attend(q, K, V):
    """q [nq, D], K and V [rows, nk, D] of one sequence."""
    g = q.shape[0] // K.shape[1]
    K, V = (t.transpose(0, 1).repeat_interleave(g, 0).contiguous() for t in (K, V))
    p = torch.softmax((K * q[:, None]).sum(-1) / math.sqrt(q.shape[1]), dim=-1)
    return (p[..., None] * V).sum(1)


def _exact_attention(c, seed):
    B, nq, nk, dim, cap = c["B"], c["nq"], c["nk"], c["dim"], c["cap"]
    i = _attention_inputs(c, seed)
    q, k, v = (t.double() for t in i["qkv"].split([nq * dim, nk * dim, nk * dim], dim=1))
    q, k, v = q.view(B, nq, dim), k.view(B, nk, dim), v.view(B, nk, dim)
    lens, starts = i["len"].tolist(), i["start"].tolist()
    kc, vc = i["kc"], i["vc"]
    if c["fused"]:
        kc, vc = kc.double(), vc.double()
        q = _rotate(_rms(q, i["wq"]), i["pos"])
        k = _rotate(_rms(k, i["wk"]), i["pos"])
        for b in range(B):
            slot = (starts[b] + lens[b] - 1) % cap
            kc[b, slot], vc[b, slot] = k[b].reshape(-1), v[b].reshape(-1)
    out = torch.empty(B, nq, dim, dtype=torch.float64, device="cuda")
    for b in range(B):
        at = (starts[b] + torch.arange(lens[b], device="cuda")) % cap
        out[b] = _attend(q[b], kc[b, at].double().view(-1, nk, dim), vc[b, at].double().view(-1, nk, dim))
    out = out.view(B, -1)
    return [out, kc, vc] if c["fused"] else [out]


def _exact_deltanet(c, seed):
    B, nkh, nvh = c["B"], c["nkh"], c["nvh"]
    i = _deltanet_inputs(c, seed)
    conv, w, x = i["conv"].double(), i["cw"].double(), i["x"].double()
    at = (i["pos"].long()[:, None] + torch.arange(3, device="cuda")) % 3
    taps = torch.gather(conv, 2, at[:, None].expand_as(conv))
    m = _silu((taps * w[:, :3]).sum(-1) + x * w[:, 3])
    conv.scatter_(2, i["pos"].long()[:, None, None].expand(B, conv.shape[1], 1), x[..., None])
    q, k, v = m.split([nkh * D, nkh * D, nvh * D], dim=1)
    unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-12)  # noqa: E731
    q, k = (unit(t.reshape(B, nkh, D)).repeat_interleave(nvh // nkh, 1) for t in (q, k))
    q, v, S = q * D ** -0.5, v.reshape(B, nvh, D), i["S"].double()
    delta = v - (S * k[..., None]).sum(2)
    S = i["decay"].double()[..., None, None] * S + i["beta"].double()[..., None, None] * k[..., None] * delta[:, :, None]
    y = _rms((S * q[..., None]).sum(2), i["nw"])
    return [(y * _silu(i["z"].double().view(B, nvh, D))).reshape(B, -1), S, conv, None]


def _exact_sample(c, seed):
    if c["temperature"] <= 0:
        return None   # token ids alone
    i = _sample_inputs(c, seed)
    rows = c["rows"]
    f = lambda v: float(np.float32(v))  # noqa: E731  -- the parameters are 32-bit floats
    seen = (torch.arange(WINDOW, device="cuda")[None] < i["hist_len"][:, None]).double()
    count = torch.zeros(rows, c["vocab"], dtype=torch.float64, device="cuda").scatter_add_(1, i["hist"].long(), seen)
    x = i["logits"].double()
    x = torch.where(count > 0, torch.where(x > 0, x / f(REP), x * f(REP)), x) - f(FREQ) * count
    return [None, torch.softmax(x / f(c["temperature"]), dim=-1)]


def _exact_decode(c, seed):
    H, nq, nk, I = MODELS["0.6b"]
    B, n = c["B"], c["context"]
    weights = _weights_06b()
    take = lambda: next(weights)[1]  # noqa: E731  -- in the checkpoint's order
    proj = lambda x, w: x @ _to_f16_down(w.double()).t().contiguous()  # noqa: E731
    embed, final = take(), take()
    pos = torch.arange(n + 1, device="cuda")
    mask = torch.full((n + 1, n + 1), -math.inf, dtype=torch.float64, device="cuda").triu_(1)
    mask[n, 0] = -math.inf   # the rings hold `context` rows: the last token has pushed out the first
    x = embed[_decode_tokens(c, seed).t().long()].double()   # [B, n + 1, H]
    for _ in range(LAYERS_06B):
        wq, wk, wv, wo, gq, gk, wg, wu, wd, w_in, w_post = (take() for _ in range(11))
        a = _rms(x, w_in)
        q = _rotate(_rms(proj(a, wq).view(B, n + 1, nq, D), gq), pos)
        k = _rotate(_rms(proj(a, wk).view(B, n + 1, nk, D), gk), pos)
        v = proj(a, wv).view(B, n + 1, nk, D)
        out = []
        for b in range(B):
            qb = q[b].transpose(0, 1).contiguous()
            kb, vb = (t[b].transpose(0, 1).repeat_interleave(nq // nk, 0).contiguous() for t in (k, v))
            p = torch.softmax(qb @ kb.transpose(1, 2).contiguous() / math.sqrt(D) + mask, dim=-1)
            out.append((p @ vb).transpose(0, 1).reshape(n + 1, -1))
        x = x + proj(torch.stack(out), wo)
        a = _rms(x, w_post)
        x = x + proj(_silu(proj(a, wg)) * proj(a, wu), wd)
    return [proj(_rms(x[:, n], final), embed)]


def _exact_convert(c, seed):
    return [_to_f16_down(_Rand(seed).normal(sum(_convert_sizes(c)), std=0.02).bfloat16().double())]
