"""The work that a user of this framework has it do, as cases that can be timed and checked.

Three ways in, all public: the fused W4A16 engine (``models.engine_for`` on a Qwen3 tree), the operator-by-operator model
(``Qwen3ModelWeek3``) and the layer-list engine (``models.engine_for`` on a layer-list checkpoint).  Each is taken in both of its
directions, prompts (prefill) and new tokens (decode), from one short sequence to many or long ones.

``listed`` / ``draw`` give cases, ``prepare`` what a program has in hand before the call, ``run`` one pass, ``work`` what the pass cannot
do without, ``exact`` its results in 64 bits from plain torch, ``tolerance`` how far a correct implementation may be from another.

Checkpoints are random with two properties of trained ones that random weights lack: the residual stream keeps a clear component of the token it
came from, and the head answers with one clear favourite (row (a t + b) mod vocabulary of the head is the embedding of token t).  Greedy
tokens are therefore the same for every correct implementation, while every logit still carries what all layers added to the stream.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
for _p in (ROOT / "tiny-llm_amd", ROOT / "tiny-llm_amd" / "extensions_hip"):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

DEV = "cuda"
PAGE = 128

QWEN = {  # sizes of the two Qwen3 configurations this framework is run on
    "qwen3-4b": dict(hidden_size=2560, num_hidden_layers=36, num_attention_heads=32, num_key_value_heads=8, head_dim=128, intermediate_size=9728,
                     vocab_size=151936, rope_theta=1000000, rms_norm_eps=1e-6, max_position_embeddings=40960, tie_word_embeddings=False),
    "qwen3-0.6b": dict(hidden_size=1024, num_hidden_layers=28, num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=3072,
                       vocab_size=151936, rope_theta=1000000, rms_norm_eps=1e-6, max_position_embeddings=40960, tie_word_embeddings=False),
}
HEAD_STEP, HEAD_SHIFT = 4099, 1237  # the favourite that follows token t: (4099 t + 1237) mod vocabulary (4099 is prime and divides none of the vocabularies)


# ---- cases ---------------------------------------------------------------------------------------------------------------------------------

def listed():
    engine = dict(path="engine", kv="bf16")
    ops = dict(path="operators", model="qwen3-4b", layers=6)
    lists = dict(path="layers", dtype="bf16")
    return [
        # one more token of a short chat on the small model: the smallest call there is, launches and latency
        dict(name="engine_decode_small", model="qwen3-0.6b", leg="decode", batch=1, context=33, steps=1, **engine),
        # a single user's answer on the 4B model behind a short prompt: the headline decode
        dict(name="engine_decode_one", model="qwen3-4b", leg="decode", batch=1, context=128, steps=16, **engine),
        # the same behind a long document
        dict(name="engine_decode_long", model="qwen3-4b", leg="decode", batch=1, context=31999, steps=8, **engine),
        # 64 users of a server at once, contexts of all lengths
        dict(name="engine_decode_many", model="qwen3-4b", leg="decode", batch=64, context=777, steps=4, **engine),
        # a long prompt, in the engine's own chunks
        dict(name="engine_prefill_long", model="qwen3-4b", leg="prefill", batch=1, context=8192, steps=0, **engine),
        # what a server admits in one turn: several short prompts of unequal length in one pass
        dict(name="engine_prefill_packed", model="qwen3-4b", leg="prefill", batch=6, context=333, steps=0, **engine),
        # the operator-by-operator model, as the reference's chapters use it: a prompt, and tokens behind it
        dict(name="operators_prefill", leg="prefill", context=1000, steps=0, **ops),
        dict(name="operators_decode", leg="decode", context=300, steps=4, **ops),
        # layer lists: a prompt in one chunk, through recurrences and attention (Fonapel), through recurrences, latent attention and experts (Zefapel)
        dict(name="fonapel_prefill", family="Fonapel", width=2048, leg="prefill", batch=1, context=2048, steps=0, **lists),
        dict(name="zefapel_prefill", family="Zefapel", width=2048, leg="prefill", batch=1, context=1900, steps=0, **lists),
        # a few requests answered together, and one alone
        dict(name="fonapel_requests", family="Fonapel", width=1024, leg="generate", batch=4, context=200, steps=48, **lists),
        dict(name="zefapel_request", family="Zefapel", width=2048, leg="generate", batch=1, context=150, steps=32, **lists),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(("engine", "engine", "operators", "layers", "layers"))
    if path == "engine":
        model = rng.choice(("qwen3-4b", "qwen3-4b", "qwen3-0.6b"))
        if rng.random() < 0.5:
            batch = _log(rng, 1, 64)
            return dict(path=path, kv=rng.choice(("bf16", "bf16", "fp8")), model=model, leg="decode", batch=batch, context=_log(rng, 16, 31999 if batch == 1 else 24000 // batch),
                        steps=rng.randint(1, 8))
        batch = rng.choice((1, 1, 1, rng.randint(2, 12)))
        return dict(path=path, kv="bf16", model=model, leg="prefill", batch=batch, context=_log(rng, 5, 8192 if batch == 1 else 2048 // batch), steps=0)
    if path == "operators":
        leg = rng.choice(("prefill", "decode"))
        return dict(path=path, model="qwen3-4b", layers=6, leg=leg, context=_log(rng, 3, 2048), steps=0 if leg == "prefill" else rng.randint(1, 4))
    family, leg = rng.choice(("Fonapel", "Zefapel")), rng.choice(("prefill", "prefill", "generate"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "float32"))
    width = rng.choice((512, 1024, 2048) if dtype == "float32" else (512, 1024, 1536, 2048, 3072))
    batch = rng.choice((1, 1, rng.randint(2, 8)))
    if leg == "generate":
        return dict(path=path, family=family, width=width, dtype=dtype, leg=leg, batch=batch, context=_log(rng, 4, 600 // batch), steps=rng.randint(8, 48))
    return dict(path=path, family=family, width=width, dtype=dtype, leg=leg, batch=batch, context=_log(rng, 9, (3000 if dtype == "bf16" else 1000) // batch), steps=0)


def _lengths(case):
    """Tokens of each sequence: unequal where there are several, from the context asked for down to a tenth of it."""
    c, b = case["context"], case.get("batch", 1)
    return [max(2, c - (i * 9 * c) // (10 * b)) for i in range(b)]


def _prompts(case, seed, vocab):
    rng = np.random.default_rng(seed)
    return [[int(t) for t in rng.integers(1, vocab, n)] for n in _lengths(case)]


# ---- checkpoints (what a user has loaded; the same for every seed) ---------------------------------------------------------------------------

_CKPT = {}


def _kept(key, make):
    """The checkpoint loaded last stays in memory, as in a program that serves one model."""
    if key not in _CKPT:
        _CKPT.clear()
        _CKPT[key] = make()
    return _CKPT[key]


def _next_row(vocab):
    return (torch.arange(vocab, dtype=torch.int64, device=DEV) * HEAD_STEP + HEAD_SHIFT) % vocab


def _qwen(model, layers=None):
    cfg = dict(QWEN[model])
    if layers:
        cfg["num_hidden_layers"] = layers

    def make():
        gen = torch.Generator(device=DEV).manual_seed(20)

        def linear(rows, cols, sigma):
            """Codes uniform in 0 .. 15, scales spread by a tenth, zero point in the middle: weights of standard deviation `sigma`."""
            words = torch.randint(-2 ** 31, 2 ** 31, (rows, cols // 8), generator=gen, device=DEV, dtype=torch.int64).to(torch.int32)
            scale = (sigma / 4.61) * (1.0 + 0.1 * torch.randn((rows, cols // 128), generator=gen, device=DEV))
            scales = scale.to(torch.bfloat16)
            return SimpleNamespace(weight=words, scales=scales, biases=(-7.5 * scales.float()).to(torch.bfloat16), group_size=128, bits=4)

        def norm(n):
            return SimpleNamespace(weight=(1.0 + 0.05 * torch.randn(n, generator=gen, device=DEV)).to(torch.bfloat16))

        h, inter, hd = cfg["hidden_size"], cfg["intermediate_size"], cfg["head_dim"]
        hq, hkv, s, out = cfg["num_attention_heads"], cfg["num_key_value_heads"], h ** -0.5, 0.15 * h ** -0.5
        blocks = [SimpleNamespace(self_attn=SimpleNamespace(q_proj=linear(hq * hd, h, s), k_proj=linear(hkv * hd, h, s), v_proj=linear(hkv * hd, h, s),
                                                            o_proj=linear(h, hq * hd, out), q_norm=norm(hd), k_norm=norm(hd)),
                                  mlp=SimpleNamespace(gate_proj=linear(inter, h, s), up_proj=linear(inter, h, s), down_proj=linear(h, inter, out)),
                                  input_layernorm=norm(h), post_attention_layernorm=norm(h)) for _ in range(cfg["num_hidden_layers"])]
        embed = linear(cfg["vocab_size"], h, 1.0)
        head = SimpleNamespace(weight=torch.empty_like(embed.weight), scales=torch.empty_like(embed.scales), biases=torch.empty_like(embed.biases), group_size=128, bits=4)
        to = _next_row(cfg["vocab_size"])
        head.weight[to], head.scales[to], head.biases[to] = embed.weight, embed.scales, embed.biases
        return SimpleNamespace(args=SimpleNamespace(**cfg), model=SimpleNamespace(embed_tokens=embed, layers=blocks, norm=norm(h)), lm_head=head)

    return _kept(("qwen", model, cfg["num_hidden_layers"]), make)


def _list_config(family, width, vocab=32768):
    """Four layers of head width 128, as this framework's own comparison of the families runs them."""
    heads, kv = width // 128, max(1, width // 512)
    if family == "Fonapel":
        ff = {"kind": "dense", "ff": 3 * width}
        attn = {"type": "attention", "mixer": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "rot": {"dims": 64, "base": 1e6}, "scale": 128 ** -0.5}, "mlp": ff}
        delta = {"type": "delta", "mixer": {"heads": heads, "kv_heads": heads, "dim": 128, "vdim": 128, "conv": 4}, "mlp": ff}
        return {"architecture": family, "layers": [delta, attn, attn, delta], "norm": {"eps": 1e-5}, "residual_mult": 0.5, "vocab": vocab, "width": width}
    dense = {"kind": "dense", "ff": 2 * width}
    moe = {"kind": "moe", "expert": {"ff": width // 2}, "router": {"experts": 8, "identity": 2, "top": 2, "groups": {"count": 5, "keep": 3}}, "shared": {"ff": width}}
    rot = {"base": 1e6, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}
    latent = {"heads": heads, "dim": 128, "vdim": 128, "rot_dim": 64, "q_rank": max(64, width // 2), "kv_rank": 192, "rot": rot, "scale": 192 ** -0.5}
    layers = [{"type": "mlstm", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "gate_cap": 20.0}, "mlp": dense},
              {"type": "gla", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "tau": 8.0}, "mlp": moe},
              {"type": "latent_attention", "mixer": dict(latent), "mlp": dense}, {"type": "latent_attention", "mixer": dict(latent, kv_from=2), "mlp": moe}]
    return {"architecture": family, "embedding": {"scale": 1.0}, "layers": layers, "norm": {"eps": 1e-6}, "vocab": vocab, "width": width}


def _layer_list(family, width):
    def make():
        from tiny_llm_hip.synthetic import synthetic_layer_list

        config = _list_config(family, width)
        model = synthetic_layer_list(config, seed=20, device=DEV)
        embed = model.tensors["embed"]
        head = torch.empty_like(embed)
        head[_next_row(config["vocab"])] = (embed.float() * (1.5 * width ** -0.5)).to(embed.dtype)
        model.tensors["head"] = head
        return config, model

    return _kept((family, width), make)


# ---- prepare and run ---------------------------------------------------------------------------------------------------------------------------

def _admit(engine, prompts, rows):
    """Begin a slot per prompt and prefill them: short ones packed into passes of at most `rows` tokens and 16 slots, long ones in chunks."""
    group, held = [], 0

    def flush():
        nonlocal group, held
        if group:
            engine.prefill_packed(group)
        group, held = [], 0

    for slot, p in enumerate(prompts):
        engine.begin(slot)
        if len(p) > rows:
            engine.prefill(slot, p)
            continue
        if held + len(p) > rows or len(group) == 16:
            flush()
        group.append((slot, p, True))
        held += len(p)
    flush()


def prepare(case, seed):
    from tiny_llm_hip.models import engine_for

    s = SimpleNamespace(case=case)
    if case["path"] == "operators":
        from tiny_llm_hip import Qwen3ModelWeek3

        s.model = Qwen3ModelWeek3(_qwen(case["model"], case["layers"]), page_size=PAGE)
        s.prompt = torch.tensor(_prompts(case, seed, s.model.vocab_size), dtype=torch.int64, device=DEV)
        s.cache = s.model.create_kv_cache()
        if case["leg"] == "decode":
            s.token = s.model(s.prompt, 0, s.cache, logits_to_keep=1).argmax(dim=-1)
        return s
    batch, lens, steps = case["batch"], _lengths(case), case["steps"]
    per_seq = [-(-(n + steps + 2) // PAGE) + 1 for n in lens]
    pool = dict(page_size=PAGE, num_pages=sum(per_seq) + 2, max_batch=batch, max_pages_per_seq=max(per_seq))
    if case["path"] == "engine":
        ckpt = _qwen(case["model"])
        s.prompts = _prompts(case, seed, ckpt.args.vocab_size)
        rows = 4096 if max(lens) > 2048 else 2048
        s.engine = engine_for(ckpt, max_prefill_rows=rows, kv_format=case["kv"], **pool)
        if case["leg"] == "decode":
            _admit(s.engine, s.prompts, rows)
            s.first = s.engine.read_pending(batch)
    else:
        config, model = _layer_list(case["family"], case["width"])
        s.prompts = _prompts(case, seed, config["vocab"])
        s.engine = engine_for(model, max_prefill_rows=max(64, sum(lens)), dtype=torch.bfloat16 if case["dtype"] == "bf16" else torch.float32, **pool)
    return s


def run(s):
    case = s.case
    leg, steps = case["leg"], case["steps"]
    if case["path"] == "operators":
        if leg == "prefill":
            logits = s.model(s.prompt, 0, s.cache, logits_to_keep=1)
            for layer in s.cache:
                layer.release()
            return {"logits": logits[:, 0]}
        token, at, tokens = s.token, s.prompt.shape[1], []
        for i in range(steps):
            logits = s.model(token, at + i, s.cache, logits_to_keep=1)
            token = logits.argmax(dim=-1)
            tokens.append(token)
        for layer in s.cache:
            layer.rewind(steps)
        return {"tokens": torch.cat(tokens, 1), "logits": logits[:, 0]}
    e, batch = s.engine, case["batch"]
    if leg == "decode":  # go on from the prompt's end, as a server's loop does: one step, then its tokens
        for slot in range(batch):
            e.set_token(slot, s.first[slot])
        if batch == 1:
            e.decode(steps, batch=1)
            tokens = np.array([e.read_tokens(0, steps)], dtype=np.int64)
        else:
            got = []
            for _ in range(steps):
                e.decode(1, batch=batch)
                got.append(e.read_pending(batch))
            tokens = np.array(got, dtype=np.int64).T
        logits = e.logits(batch)
        for slot in range(batch):
            e.rewind(slot, steps)
        return {"tokens": tokens, "logits": logits}
    if batch == 1:
        e.begin(0)
        e.prefill(0, s.prompts[0])
    else:
        for slot in range(batch):
            e.begin(slot)
        e.prefill_packed([(slot, p, True) for slot, p in enumerate(s.prompts)])
    if leg == "generate":
        e.decode(steps, batch=batch)
        tokens = [e.read_tokens(slot, steps + 1) for slot in range(batch)]
    else:
        tokens = [[t] for t in e.read_pending(batch)]
    logits = e.logits(batch)
    for slot in range(batch):
        e.release(slot)
    return {"tokens": np.array(tokens, dtype=np.int64), "logits": logits}


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------------------------------

def _pairs(n, new):
    """(query, key) pairs of `new` queries at the end of a causal sequence of n."""
    return new * n - new * (new - 1) // 2


def work(case):
    lens, steps = _lengths(case), case["steps"]
    if case["path"] in ("engine", "operators"):
        c = QWEN[case["model"]]
        n_layers = case.get("layers") or c["num_hidden_layers"]
        h, hq, hkv, d, inter, v = (c[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size", "vocab_size"))
        mats = n_layers * (h * (hq + 2 * hkv) * d + hq * d * h + 3 * h * inter)
        w4 = 0.5 + 4 / 128
        row = n_layers * hkv * (2 * (d + 4) if case.get("kv") == "fp8" else 4 * d)  # bytes of one token's keys and values
        pair = n_layers * hq * 4 * d
        if case["leg"] == "decode":
            kv = sum(n * steps + steps * (steps + 1) // 2 for n in lens)
            return {"bytes": steps * ((mats + v * h) * w4 + len(lens) * v * 2) + kv * row, "flops": 2 * steps * len(lens) * (mats + v * h) + kv * pair}
        tokens = sum(lens)
        return {"bytes": (mats + v * h) * w4 + tokens * row + len(lens) * v * 2, "flops": 2 * (tokens * mats + len(lens) * v * h) + pair * sum(_pairs(n, n) for n in lens)}
    config = _list_config(case["family"], case["width"])
    W, item = config["width"], 2 if case["dtype"] == "bf16" else 4
    fixed, taken, pair, row, state, rec = 0, [], 0, 0, 0, 0
    for L in config["layers"]:
        m, mlp = L["mixer"], L["mlp"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        fixed += H * V * W
        if L["type"] == "attention":
            G = m["kv_heads"]
            fixed += W * (H * D + G * (D + V) + H * V)
            pair += 2 * H * (D + V)
            row += G * (D + V) * item
        elif L["type"] == "latent_attention":
            R, C, Q = m["rot_dim"], m["kv_rank"], m["q_rank"]
            fixed += W * Q + Q * H * (D + R) + H * (D + V) * C + H * V * W + (0 if "kv_from" in m else W * (C + R))
            pair += 2 * H * (D + R + V)
            row += 0 if "kv_from" in m else (C + R) * item
        else:  # recurrences: read, decay, write and read out a state of D x V a head and token
            gates = {"delta": 2 * H, "mlstm": 2 * H, "gla": 16}[L["type"]]
            fixed += W * (2 * H * D + 2 * H * V + gates) + (16 * H * D if L["type"] == "gla" else 0)
            state += 4 * H * D * V
            rec += H * D * V * (8 if L["type"] == "delta" else 5)
        if mlp["kind"] == "dense":
            fixed += (2 if case["family"] == "Fonapel" else 3) * W * mlp["ff"]
        else:
            r = mlp["router"]
            fixed += W * (r["experts"] + r["identity"]) + 2 * W * mlp["shared"]["ff"] + W
            taken.append((2 * W * mlp["expert"]["ff"], r["top"], r["experts"]))
    head = config["vocab"] * W

    def one(tokens, seqs, pairs):
        experts_read = sum(e * min(n, top * tokens) for e, top, n in taken)
        return ((fixed + experts_read + head) * item + 2 * seqs * state + seqs * config["vocab"] * 4 + tokens * row,
                2 * tokens * (fixed + sum(e * top for e, top, _ in taken)) + 2 * seqs * head + pairs * pair + tokens * rec)

    nbytes, flops = one(sum(lens), len(lens), sum(_pairs(n, n) for n in lens))
    for i in range(steps if case["leg"] == "generate" else 0):
        b, f = one(len(lens), len(lens), sum(n + i + 1 for n in lens))
        nbytes, flops = nbytes + b + sum(n + i for n in lens) * row, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Logits, against another correct implementation at the same precision (the greedy tokens have to be the same).  Seen against 64 bits: up to 3.5e-6 in
    float32, 0.002 .. 0.005 for a layer list in bf16 (float32 stream, four layers), 0.007 through six and 0.014 .. 0.022 through 28 or 36 layers with a bf16 stream."""
    if case["path"] == "layers":
        return {"rel": 2e-5, "max": 5e-4} if case["dtype"] == "float32" else {"rel": 1.5e-2, "max": 0.1}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------------------------------------

def _greedy(forward, prompts, steps, vocab):
    """(tokens [b][1 + steps], logits [b, vocab] behind the last) of a model given by ``forward(sequences, keep)`` = logits [b, keep, vocab] of the last `keep`
    rows: guess the answers, score them in one pass, correct the first wrong token of each and score again until all are the model's own."""
    answers = []
    for p in prompts:
        a, t = [], p[-1]
        for _ in range(steps):
            t = (t * HEAD_STEP + HEAD_SHIFT) % vocab
            a.append(t)
        answers.append(a)
    while True:
        logits = forward([p + a for p, a in zip(prompts, answers)], steps + 1)
        best = logits.argmax(-1).tolist()
        wrong = False
        for a, b in zip(answers, best):
            for i in range(steps):
                if a[i] != b[i]:
                    a[i], wrong = b[i], True
                    break
        if not wrong:
            return best, logits[:, -1]


def _rms(x, w, eps):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _causal(q, k, v, scale, sink=False, block=2048):
    """q [L, H, D], k [L, G, D], v [L, G, V] -> [L, H V]: ordinary softmax, or with a 1 in the denominator, a block of queries at a time."""
    L, H, _ = q.shape
    G, out = k.shape[1], []
    block = max(64, min(block, int(3e8) // max(1, L)))
    k, v = k.permute(1, 2, 0), v.transpose(0, 1)
    for g in range(G):
        rows = []
        for i in range(0, L, block):
            n = min(L, i + block)
            s = (q[i:n, g * (H // G):(g + 1) * (H // G)].transpose(0, 1) @ k[g, :, :n]) * scale
            s.masked_fill_(torch.ones(n - i, n, dtype=torch.bool, device=s.device).triu_(i + 1), float("-inf"))
            top = s.amax(-1, keepdim=True).clamp_(min=0.0) if sink else s.amax(-1, keepdim=True)
            s = s.sub_(top).exp_()
            rows.append((s @ v[g, :n]) / (s.sum(-1, keepdim=True) + (torch.exp(-top) if sink else 0.0)))
        out.append(torch.cat(rows, 1))
    return torch.cat(out, 0).transpose(0, 1).reshape(L, -1)


def _w4(q):
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device=DEV)
    codes = ((q.weight[..., None] >> shifts) & 15).reshape(q.weight.shape[0], -1, 128).double()
    return (codes * q.scales.double()[..., None] + q.biases.double()[..., None]).reshape(q.weight.shape[0], -1)


def _fp8_rows(x):
    """Rows over the last axis as E4M3 codes under one power of two each, as such a cache holds them."""
    top = x.abs().amax(-1, keepdim=True)
    scale = torch.exp2(torch.ceil(torch.log2(torch.clamp(top, min=2.0 ** -100) / 448.0)))
    return (x / scale).to(torch.bfloat16).to(torch.float8_e4m3fn).double() * scale


def _qwen_forward(ckpt, kv):
    c = ckpt.args

    def forward(seqs, keep):
        bounds = np.cumsum([0] + [len(s) for s in seqs]).tolist()
        ids = torch.tensor([t for s in seqs for t in s], device=DEV)
        pos = torch.cat([torch.arange(len(s), device=DEV) for s in seqs]).double()
        e = ckpt.model.embed_tokens
        x = _w4(SimpleNamespace(weight=e.weight[ids], scales=e.scales[ids], biases=e.biases[ids]))
        d, half = c.head_dim, c.head_dim // 2
        angle = pos[:, None] * (float(c.rope_theta) ** (-torch.arange(half, device=DEV).double() / half))
        cos, sin = angle.cos()[:, None], angle.sin()[:, None]

        def turn(z):
            a, b = z[..., :half], z[..., half:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

        for layer in ckpt.model.layers:
            at, ml = layer.self_attn, layer.mlp
            y = _rms(x, layer.input_layernorm.weight.double(), c.rms_norm_eps)
            q = turn(_rms((y @ _w4(at.q_proj).T).unflatten(-1, (-1, d)), at.q_norm.weight.double(), c.rms_norm_eps))
            k = turn(_rms((y @ _w4(at.k_proj).T).unflatten(-1, (-1, d)), at.k_norm.weight.double(), c.rms_norm_eps))
            v = (y @ _w4(at.v_proj).T).unflatten(-1, (-1, d))
            if kv == "fp8":
                k, v = _fp8_rows(k), _fp8_rows(v)
            o = torch.cat([_causal(q[a:b], k[a:b], v[a:b], d ** -0.5) for a, b in zip(bounds, bounds[1:])])
            x = x + o @ _w4(at.o_proj).T
            y = _rms(x, layer.post_attention_layernorm.weight.double(), c.rms_norm_eps)
            x = x + (torch.nn.functional.silu(y @ _w4(ml.gate_proj).T) * (y @ _w4(ml.up_proj).T)) @ _w4(ml.down_proj).T
        rows = torch.cat([torch.arange(b - keep, b, device=DEV) for b in bounds[1:]])
        y = _rms(x[rows], ckpt.model.norm.weight.double(), c.rms_norm_eps)
        return (y @ _w4(ckpt.lm_head).T).reshape(len(seqs), keep, -1)

    return forward


def _conv_silu(z, w):
    L, taps = z.shape[0], w.shape[1]
    padded = torch.cat([z.new_zeros(taps - 1, z.shape[1]), z])
    return torch.nn.functional.silu(sum(w[:, j] * padded[j:j + L] for j in range(taps)))


def _pairwise(z, angle, mult=1.0):
    """z [L, heads, dim]: dimensions (2 i, 2 i + 1) turned by angle[:, i]; those behind pass."""
    n = angle.shape[1]
    c, s = (angle.cos() * mult)[:, None], (angle.sin() * mult)[:, None]
    u, v = z[..., 0:2 * n:2], z[..., 1:2 * n:2]
    return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), z[..., 2 * n:]], -1)


def _fonapel_mixer(h, mc, kind, t, eps):
    L, H, G, D, V = h.shape[0], mc["heads"], mc["kv_heads"], mc["dim"], mc["vdim"]
    gate = h @ t("mix.g").T
    if kind == "attention":
        n = mc["rot"]["dims"] // 2
        angle = torch.arange(L, device=DEV).double()[:, None] * (mc["rot"]["base"] ** (-torch.arange(n, device=DEV).double() / n))
        q, k = (_rms(_pairwise((h @ t(w).T).reshape(L, -1, D), angle), None, eps) for w in ("mix.q", "mix.k"))
        return _causal(q, k, (h @ t("mix.v").T).reshape(L, G, V), mc["scale"], sink=True) * torch.sigmoid(gate)
    q, k, v = (_conv_silu(h @ t(w).T, t(w + ".conv")) for w in ("mix.q", "mix.k", "mix.v"))
    q, k = (z.reshape(L, G, D) for z in (q, k))
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    q, k, v = q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1), v.reshape(L, H, V)
    beta = torch.sigmoid(h @ t("mix.b").T)
    g = torch.exp(-torch.exp(t("mix.A_log")) * torch.nn.functional.softplus(h @ t("mix.a").T + t("mix.dt_bias")))
    state, out = h.new_zeros(H, D, V), h.new_empty(L, H, V)
    for i in range(L):
        state = state * g[i, :, None, None]
        u = beta[i, :, None] * (v[i] - (k[i, :, None] @ state)[:, 0])
        state = torch.baddbmm(state, k[i, :, :, None], u[:, None])
        out[i] = (q[i, :, None] @ state)[:, 0]
    return _rms(out, t("mix.norm"), eps).reshape(L, H * V) * torch.nn.functional.silu(gate)


def _zefapel_mixer(h, mc, kind, t, eps, latents, index):
    L, H, D, V = h.shape[0], mc["heads"], mc["dim"], mc["vdim"]
    sigmoid, logsigmoid = torch.sigmoid, torch.nn.functional.logsigmoid
    gate = h @ t("mix.g").T
    if kind == "latent_attention":
        R, C, rot = mc["rot_dim"], mc["kv_rank"], mc["rot"]
        n, base, sc = rot["dims"] // 2, rot["base"], rot["scaling"]
        f = base ** (-torch.arange(n, device=DEV).double() / n)
        at = [2 * n * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base)) for turns in (sc["fast"], sc["slow"])]
        lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), 2 * n - 1)
        ramp = ((torch.arange(n, device=DEV).double() - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        angle = torch.arange(L, device=DEV).double()[:, None] * (f / sc["factor"] * ramp + f * (1 - ramp))
        mult = 0.1 * math.log(sc["factor"]) + 1.0
        q = (_rms(h @ t("mix.dq").T, t("mix.dq.norm"), eps) @ t("mix.uq").T).reshape(L, H, D + R)
        if "kv_from" in mc:
            c, k_rot = latents[mc["kv_from"]]
        else:
            dkv = h @ t("mix.dkv").T
            c, k_rot = latents[index] = _rms(dkv[:, :C], t("mix.dkv.norm"), eps), _pairwise(dkv[:, None, C:], angle, mult)
        q = torch.cat([q[..., :D], _pairwise(q[..., D:], angle, mult)], -1)
        k = torch.cat([(c @ t("mix.uk").T).reshape(L, H, D), k_rot.expand(L, H, R)], -1)
        return _causal(q, k, (c @ t("mix.uv").T).reshape(L, H, V), mc["scale"]) * sigmoid(gate)
    q, k, v = (h @ t("mix.q").T).reshape(L, H, D) * D ** -0.5, (h @ t("mix.k").T).reshape(L, H, D), (h @ t("mix.v").T).reshape(L, H, V)
    state, out = h.new_zeros(H, D, V), h.new_empty(L, H, V)
    if kind == "gla":
        alpha = torch.exp(logsigmoid((h @ t("mix.a1").T) @ t("mix.a2").T + t("mix.a2.b")) / mc["tau"]).reshape(L, H, D)
        for i in range(L):
            state = torch.baddbmm(state * alpha[i, :, :, None], k[i, :, :, None], v[i, :, None])
            out[i] = (q[i, :, None] @ state)[:, 0]
        return _rms(out, t("mix.norm"), eps).reshape(L, H * V) * torch.nn.functional.silu(gate)
    cap = mc["gate_cap"]
    li = cap * torch.tanh((h @ t("mix.i").T + t("mix.i.b")) / cap)
    lf = logsigmoid(cap * torch.tanh((h @ t("mix.f").T + t("mix.f.b")) / cap))
    n, m = h.new_zeros(H, D), h.new_zeros(H)
    for i in range(L):
        top = torch.maximum(lf[i] + m, li[i])
        a, b = torch.exp(lf[i] + m - top), torch.exp(li[i] - top)
        state = torch.baddbmm(state * a[:, None, None], k[i, :, :, None] * b[:, None, None], v[i, :, None])
        n, m = n * a[:, None] + k[i] * b[:, None], top
        low = torch.maximum((n * q[i]).sum(-1).abs(), torch.exp(-m)) + 1e-6
        out[i] = (q[i, :, None] @ state)[:, 0] / low[:, None]
    return _rms(out, None, eps).reshape(L, H * V) * t("mix.norm") * sigmoid(gate)


def _zefapel_ff(h, mlp, t):
    if mlp["kind"] == "dense":
        return (torch.nn.functional.silu(h @ t("mlp.gate").T) * (h @ t("mlp.up").T)) @ t("mlp.down").T
    r = mlp["router"]
    score = torch.softmax(h @ t("mlp.router").T, -1)
    choice = score + t("mlp.correction")
    groups = choice.unflatten(-1, (r["groups"]["count"], -1))
    kept = torch.zeros_like(groups[..., 0]).scatter_(-1, groups.amax(-1).topk(r["groups"]["keep"], -1).indices, 1.0)
    choice = torch.where(kept[..., None] > 0, groups, torch.full_like(groups, float("-inf"))).flatten(-2)
    weight = torch.zeros_like(score).scatter_(-1, choice.topk(r["top"], -1).indices, 1.0) * score
    out = h * weight[:, r["experts"]:].sum(-1, keepdim=True)
    for j in range(r["experts"]):
        out = out + weight[:, j:j + 1] * (torch.relu(h @ t(f"mlp.e{j}.up").T) ** 2 @ t(f"mlp.e{j}.down").T)
    return out + (torch.relu(h @ t("mlp.shared.up").T) ** 2 @ t("mlp.shared.down").T) * torch.sigmoid(h @ t("mlp.shared.sg").T)


def _list_forward(config, tensors):
    fonapel = config["architecture"] == "Fonapel"
    eps = config["norm"]["eps"]

    def dyt(x, name):
        return torch.tanh(tensors[name + ".alpha"].double() * x) * tensors[name].double() + tensors[name + ".b"].double()

    def one(seq, keep):
        x, latents = tensors["embed"][torch.tensor(seq, device=DEV)].double(), {}
        for i, L in enumerate(config["layers"]):
            def t(name, p=f"l{i}."):
                return tensors[p + name].double()

            if fonapel:
                h = _rms(x, 1.0 + t("norm1"), eps)
                y = _fonapel_mixer(h, L["mixer"], L["type"], t, eps) @ t("mix.o").T
                x = x + config["residual_mult"] * (y + torch.nn.functional.gelu(h @ t("mlp.up").T) @ t("mlp.down").T)
            else:
                x = x + t("ls1") * (_zefapel_mixer(dyt(x, f"l{i}.norm1"), L["mixer"], L["type"], t, eps, latents, i) @ t("mix.o").T)
                x = x + t("ls2") * _zefapel_ff(dyt(x, f"l{i}.norm2"), L["mlp"], t)
        y = _rms(x[-keep:], 1.0 + tensors["final.norm"].double(), eps) if fonapel else dyt(x[-keep:], "final.norm")
        return y @ tensors["head"].double().T

    return lambda seqs, keep: torch.stack([one(s, keep) for s in seqs])


def exact(case, seed):
    if case["context"] > 24000:  # (half a minute of 64-bit products)
        return None
    if case["path"] == "layers":
        config, model = _layer_list(case["family"], case["width"])
        prompts, forward = _prompts(case, seed, config["vocab"]), _list_forward(config, model.tensors)
    else:
        ckpt = _qwen(case["model"], case.get("layers"))
        prompts, forward = _prompts(case, seed, ckpt.args.vocab_size), _qwen_forward(ckpt, case.get("kv"))
    vocab = config["vocab"] if case["path"] == "layers" else ckpt.args.vocab_size
    tokens, logits = _greedy(forward, prompts, case["steps"], vocab)
    if case["path"] == "operators" and case["leg"] == "prefill":
        return {"logits": logits}
    tokens = np.array(tokens, dtype=np.int64)
    return {"tokens": tokens[:, 1:] if case["leg"] == "decode" else tokens, "logits": logits}
