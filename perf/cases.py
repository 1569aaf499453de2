"""The work that a user has the engine do, as measured cases: steps of the model runner (``ModelRunner.step``, what the
engine, the trace replay and the benchmark drive) with given token ids, so that every case has logits to compare.

Ranges.  Qwen3 dense decoders of the widths 1024 to 4096 and 8 to 36 layers, bfloat16: decoding 1 to 96 requests with
contexts of 16 to 1500 tokens, even and uneven; prompts of 1 to 2048 tokens, alone and several in a step; portions of a
prompt beside requests that decode.  The same in float32 (the engine's true 32-bit mode) at the narrower widths.  Balelorn
(experts named by token id, attention in chunks), Sodedra (matrix memories, a delta rule, windows) and Sefevik (latent
attention, minimal recurrences) of the widths 1024 to 4096 in bfloat16: prompts, decoding, and whole requests, prompt and
decoding together.  Layer sizes are those of ``bench.py``; pages hold 16 tokens, as the engine's default has it.

A decoding pass runs one step and then counts its token as not cached again (``CacheManager.rewind``), so that every pass
does the same work.  Models that keep a state of fixed size cannot step back: their cases run whole requests.
"""
import math

import torch

DEVICE = "cuda:0"
PAGE = 16
VOCAB_QWEN, VOCAB_DESIGN = 151936, 32768
MOST_TOKENS = 16384          # of one step, the engine's default
MODEL_LEN = 4096             # most tokens of one request, the engine's default

#: width -> (layers, query heads, feed-forward, tied head) of the Qwen3 sizes; 8 kv heads of 128
QWEN = {1024: (28, 16, 3072, True), 2048: (28, 16, 6144, True), 2560: (36, 32, 9728, True), 4096: (36, 32, 12288, False)}


def listed():
    return [
        # one user chatting with a small model: every kernel is short, launches and round trips decide
        dict(name="qwen-0.6b/1-decoding", family="qwen", width=1024, layers=28, dtype="bfloat16", kind="decode", requests=1, shortest=500, longest=500),
        # the benchmark's headline: eight requests in the middle of their answers
        dict(name="qwen-8b/8-decoding", family="qwen", width=4096, layers=36, dtype="bfloat16", kind="decode", requests=8, shortest=1152, longest=1152),
        # a busy server: many requests of uneven lengths
        dict(name="qwen-4b/64-decoding", family="qwen", width=2560, layers=36, dtype="bfloat16", kind="decode", requests=64, shortest=100, longest=1300),
        # a long prompt, one portion of the engine's default size
        dict(name="qwen-8b/prompt", family="qwen", width=4096, layers=36, dtype="bfloat16", kind="prompt", requests=1, shortest=2048, longest=2048),
        # several short questions that arrive together, sizes multiples of nothing
        dict(name="qwen-1.7b/6-prompts", family="qwen", width=2048, layers=28, dtype="bfloat16", kind="prompt", requests=6, shortest=19, longest=433),
        # continuous batching: a portion of a new prompt in one step with requests that decode
        dict(name="qwen-4b/portion-and-20", family="qwen", width=2560, layers=36, dtype="bfloat16", kind="mixed", requests=20, shortest=60, longest=700, portion=389),
        # the 32-bit mode, which checks and offline scoring run in: a prompt, and decoding
        dict(name="qwen-0.6b-f32/prompt", family="qwen", width=1024, layers=28, dtype="float32", kind="prompt", requests=1, shortest=611, longest=611),
        dict(name="qwen-1.7b-f32/4-decoding", family="qwen", width=2048, layers=28, dtype="float32", kind="decode", requests=4, shortest=300, longest=420),
        # mixtures of experts: a prompt, whose tokens use every expert, and decoding, where most experts have one or two
        dict(name="balelorn-2048/prompt", family="balelorn", width=2048, layers=8, dtype="bfloat16", kind="prompt", requests=1, shortest=2011, longest=2011),
        dict(name="balelorn-4096/12-decoding", family="balelorn", width=4096, layers=8, dtype="bfloat16", kind="decode", requests=12, shortest=40, longest=800),
        # recurrences: a prompt through matrix memories and the delta rule
        dict(name="sodedra-2048/prompt", family="sodedra", width=2048, layers=8, dtype="bfloat16", kind="prompt", requests=1, shortest=1500, longest=1500),
        # whole requests, prompts and answers, through latent attention and minimal recurrences
        dict(name="sefevik-2048/5-whole", family="sefevik", width=2048, layers=8, dtype="bfloat16", kind="whole", requests=5, shortest=60, longest=500, steps=24),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    family = rng.choices(["qwen", "balelorn", "sodedra", "sefevik"], [7, 2, 1, 1])[0]
    c = dict(family=family, dtype="bfloat16")
    if family == "qwen":
        c["kind"] = rng.choices(["decode", "prompt", "mixed"], [4, 3, 2])[0]
        if rng.random() < 0.3:
            c.update(dtype="float32", width=rng.choice([1024, 2048]))
        else:
            c["width"] = rng.choice([1024, 2048, 2560, 4096])
        c["layers"] = rng.randint(8, QWEN[c["width"]][0])
    else:
        c["kind"] = {"balelorn": rng.choice(["decode", "prompt", "mixed"]), "sodedra": rng.choice(["prompt", "whole"]), "sefevik": rng.choice(["prompt", "whole"])}[family]
        c["width"] = rng.choice([1024, 2048, 4096] if family == "balelorn" else [1024, 2048])
        c["layers"] = 4 * rng.randint(1, 2)
    f32 = c["dtype"] == "float32"
    if c["kind"] in ("decode", "mixed"):
        c["longest"] = log(16, 400 if f32 else 1500)
        c["shortest"] = c["longest"] if rng.random() < 0.4 else rng.randint(max(1, c["longest"] // 10), c["longest"])
        c["requests"] = min(log(1, 32 if f32 else 96), 48000 // c["longest"])
        if c["kind"] == "mixed":
            c["portion"] = log(16, 400 if f32 else 1200)
    elif c["kind"] == "prompt":
        c["requests"] = 1 if rng.random() < 0.5 else rng.randint(2, 6)
        c["longest"] = log(1, 700 if f32 else 2048) if c["requests"] == 1 else log(8, 120 if f32 else 340)
        c["shortest"] = c["longest"] if c["requests"] == 1 else rng.randint(max(1, c["longest"] // 10), c["longest"])
    else:
        c["requests"] = log(1, 12)
        c["longest"] = log(8, 1800 // c["requests"])
        c["shortest"] = rng.randint(max(1, c["longest"] // 10), c["longest"])
        c["steps"] = rng.randint(6, 32)
    return c


# ---- the models: configuration and tensors ------------------------------------------------------------------------------
def config_of(case):
    width, layers = case["width"], case["layers"]
    heads = max(1, width // 128)
    if case["family"] == "qwen":
        _, q_heads, ff, tied = QWEN[width]
        return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", hidden_act="silu", num_hidden_layers=layers, hidden_size=width,
                    num_attention_heads=q_heads, num_key_value_heads=8, head_dim=128, intermediate_size=ff, vocab_size=VOCAB_QWEN,
                    rope_theta=1000000.0, rms_norm_eps=1e-6, tie_word_embeddings=tied, max_position_embeddings=40960)
    if case["family"] == "balelorn":
        # attention in chunks of 1536 positions, every fourth layer over everything; one dense feed-forward in four, else 32 experts
        att = dict(heads=heads, kv_heads=max(1, heads // 4), dim=128, vdim=128, scale=128 ** -0.5, mask=dict(size=1536), v_mix=True, rot=dict(base=10000.0, dims=64))
        dense = dict(kind="dense", ff=3 * width)
        moe = dict(kind="moe", expert=dict(ff=3 * width // 4, limit=7.0), router=dict(experts=32, top=4))
        out = [dict(type="attention", mixer=dict(att, mask=None) if i % 4 == 3 else dict(att), mlp=dense if i % 4 == 0 else moe) for i in range(layers)]
        return dict(architecture="Balelorn", vocab=VOCAB_DESIGN, width=width, norm=dict(eps=1e-5), layers=out)
    if case["family"] == "sodedra":
        # of every four layers a matrix memory, an attention under a window, a delta rule and an attention; dense feed-forwards
        rot = dict(base=500000.0, dims=64, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192))
        att = dict(heads=heads, kv_heads=max(1, heads // 4), dim=128, vdim=128, scale=128 ** -0.5, mask=dict(size=1024), rot=rot)
        kinds = [dict(type="mlstm", mixer=dict(heads=max(1, heads // 2), dim=128, vdim=256, gate_cap=16.0)),
                 dict(type="attention", mixer=att),
                 dict(type="channel_delta", mixer=dict(heads=heads, kv_heads=max(1, heads // 2), dim=128, vdim=128, conv=4, decay_rank=128, gate_rank=128)),
                 dict(type="attention", mixer=att)]
        out = [dict(kinds[i % 4], mlp=dict(kind="dense", ff=3 * width)) for i in range(layers)]
        return dict(architecture="Sodedra", vocab=VOCAB_DESIGN, width=width, norm=dict(eps=1e-6), embedding=dict(scale=1.0), layers=out)
    # Sefevik: of every four layers a latent attention with rows of its own, two recurrences and one that reads the first one's rows
    rot = dict(base=10000.0, dims=64, scaling=dict(factor=8.0, original=4096, fast=16.0, slow=2.0))
    att = dict(heads=heads, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, mask=dict(size=1024), rot=rot)
    out = []
    for i in range(layers):
        mlp = dict(kind="dense", ff=3 * width)
        if i % 4 in (1, 2):
            out.append(dict(type="mingru", mixer=dict(width=width), mlp=mlp))
        else:
            out.append(dict(type="latent_attention", mixer=dict(att) if i % 4 == 0 else dict(att, kv_from=i - 3), mlp=mlp))
    return dict(architecture="Sefevik", vocab=VOCAB_DESIGN, width=width, norm=dict(eps=1e-6),
                embedding=dict(bigram=dict(buckets=65521, mul_prev=37, mul_cur=11)), layers=out)


def tensor_list(case):
    """(name, shape, how it is drawn) of every tensor of the model."""
    cfg, width = config_of(case), case["width"]
    out = []
    if case["family"] == "qwen":
        q, kv, ff = cfg["num_attention_heads"] * 128, 1024, cfg["intermediate_size"]
        out.append(("model.embed_tokens.weight", (VOCAB_QWEN, width), "wide"))
        for i in range(case["layers"]):
            at = "model.layers.%d." % i
            out += [(at + "input_layernorm.weight", (width,), "norm"), (at + "post_attention_layernorm.weight", (width,), "norm"),
                    (at + "self_attn.q_norm.weight", (128,), "norm"), (at + "self_attn.k_norm.weight", (128,), "norm"),
                    (at + "self_attn.q_proj.weight", (q, width), "matrix"), (at + "self_attn.k_proj.weight", (kv, width), "matrix"),
                    (at + "self_attn.v_proj.weight", (kv, width), "matrix"), (at + "self_attn.o_proj.weight", (width, q), "out"),
                    (at + "mlp.gate_proj.weight", (ff, width), "matrix"), (at + "mlp.up_proj.weight", (ff, width), "matrix"),
                    (at + "mlp.down_proj.weight", (width, ff), "out")]
        out.append(("model.norm.weight", (width,), "norm"))
        if not cfg["tie_word_embeddings"]:
            out.append(("lm_head.weight", (VOCAB_QWEN, width), "matrix"))
        return out
    out.append(("embed", (VOCAB_DESIGN, width), "matrix" if case["family"] == "balelorn" else "wide"))
    if case["family"] == "balelorn":
        out.append(("embed.norm", (width,), "norm"))
    if case["family"] == "sefevik":
        out.append(("bigram", (cfg["embedding"]["bigram"]["buckets"] + 1, width), "wide"))
    for i, layer in enumerate(cfg["layers"]):
        at, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        mix = at + "mix."
        if case["family"] == "balelorn":
            out += [(at + n, (width,), "norm") for n in ("norm1", "norm2", "norm1b", "norm2b")] + [(at + n, (width,), "share") for n in ("ls1", "ls2")]
            q, kv = m["heads"] * 128, m["kv_heads"] * 128
            out += [(mix + "q", (q, width), "matrix"), (mix + "k", (kv, width), "matrix"), (mix + "v", (kv, width), "matrix"),
                    (mix + "o", (width, q), "matrix"), (mix + "g", (q, width), "matrix"), (mix + "sink", (m["heads"],), "bias"), (mix + "vmix", (), "share")]
        elif layer["type"] == "attention":
            q, kv = m["heads"] * 128, m["kv_heads"] * 128
            out += [(mix + "q", (q, width), "matrix"), (mix + "k", (kv, width), "matrix"), (mix + "v", (kv, width), "matrix"), (mix + "o", (width, q), "out"),
                    (mix + "g", (q, width), "matrix"), (mix + "q.b", (q,), "bias"), (mix + "k.b", (kv,), "bias"), (mix + "v.b", (kv,), "bias")]
        elif layer["type"] == "mlstm":
            qk, v, H = m["heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
            out += [(mix + "q", (qk, width), "matrix"), (mix + "k", (qk, width), "matrix"), (mix + "v", (v, width), "matrix"), (mix + "g", (v, width), "matrix"),
                    (mix + "o", (width, v), "out"), (mix + "norm", (v,), "norm"), (mix + "i", (H, width), "matrix"), (mix + "i.b", (H,), "bias"),
                    (mix + "f", (H, width), "matrix"), (mix + "f.b", (H,), "forget")]
        elif layer["type"] == "channel_delta":
            qk, v, H = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
            out += [(mix + "q", (qk, width), "matrix"), (mix + "k", (qk, width), "matrix"), (mix + "v", (v, width), "matrix"), (mix + "b", (H, width), "matrix"),
                    (mix + "a1", (m["decay_rank"], width), "matrix"), (mix + "g1", (m["gate_rank"], width), "matrix"), (mix + "a2", (H * m["dim"], m["decay_rank"]), "matrix"),
                    (mix + "g2", (v, m["gate_rank"]), "matrix"), (mix + "o", (width, v), "out"), (mix + "q.conv", (qk, m["conv"]), "taps"),
                    (mix + "k.conv", (qk, m["conv"]), "taps"), (mix + "v.conv", (v, m["conv"]), "taps"), (mix + "A_log", (H,), "rate"),
                    (mix + "dt_bias", (H * m["dim"],), "pace"), (mix + "norm", (m["vdim"],), "norm")]
        elif layer["type"] == "mingru":
            w = m["width"]
            out += [(mix + "z", (w, width), "matrix"), (mix + "z.b", (w,), "bias"), (mix + "x", (w, width), "matrix"), (mix + "x.b", (w,), "bias"),
                    (mix + "g", (w, width), "matrix"), (mix + "o", (width, w), "matrix")]
        else:
            H, r = m["heads"], m["kv_rank"]
            out.append((mix + "q", (H * 192, width), "matrix"))
            if "kv_from" not in m:
                out += [(mix + "dkv", (r + 64, width), "matrix"), (mix + "dkv.norm", (r,), "norm")]
            out += [(mix + "uk", (H * 128, r), "matrix"), (mix + "uv", (H * 128, r), "matrix"), (mix + "sink", (H,), "bias"), (mix + "o", (width, H * 128), "matrix")]
        if case["family"] == "sodedra":
            out.append((at + "norm1", (width,), "bias"))
        if case["family"] == "sefevik":
            out += [(at + "norm1", (width,), "norm"), (at + "norm2", (width,), "norm"), (at + "dwa", (i + 2,), "mix"), (at + "mlp.act", (2,), "bias"),
                    (at + "mlp.up", (mlp["ff"], width), "matrix"), (at + "mlp.down", (width, mlp["ff"]), "matrix")]
        elif mlp["kind"] == "dense":
            out += [(at + "mlp.gate", (mlp["ff"], width), "matrix"), (at + "mlp.up", (mlp["ff"], width), "matrix"),
                    (at + "mlp.down", (width, mlp["ff"]), "out" if case["family"] == "sodedra" else "matrix")]
        else:
            f = mlp["expert"]["ff"]
            out.append((at + "mlp.table", (VOCAB_DESIGN, mlp["router"]["top"]), "table"))
            for e in range(mlp["router"]["experts"]):
                out += [(at + "mlp.e%d.gate" % e, (f, width), "matrix"), (at + "mlp.e%d.up" % e, (f, width), "matrix"), (at + "mlp.e%d.down" % e, (width, f), "matrix")]
    out.append(("final.norm", (width,), "bias" if case["family"] == "sodedra" else "norm"))
    if case["family"] != "sodedra":
        out.append(("head", (VOCAB_DESIGN, width), "matrix"))
    return out


def tensors_of(case, seed):
    """The model's tensors as a checkpoint holds them (bfloat16; widened for float32 runs), made on the device."""
    g = torch.Generator(device=DEVICE).manual_seed(2 * int(seed) + 1)
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    out = {}
    for name, shape, how in tensor_list(case):
        if how in ("matrix", "out", "wide"):
            # what writes into the stream is scaled by the depth, as initialisations have it: layers move the stream and do not replace it
            std = {"matrix": 0.02, "out": 0.02 / math.sqrt(2.0 * case["layers"]), "wide": 1.0}[how]
            t = torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(0.0, std, generator=g)
        elif how == "table":
            t = torch.rand((shape[0], 32), generator=g, device=DEVICE).argsort(dim=-1)[:, :shape[1]].to(torch.int32).contiguous()
        else:
            n, u = torch.randn(shape, generator=g, device=DEVICE), torch.rand(shape, generator=g, device=DEVICE)
            t = {"norm": lambda: 1.0 + 0.1 * n, "bias": lambda: 0.05 * n, "share": lambda: 0.3 + 0.1 * u, "taps": lambda: 0.4 * n,
                 "mix": lambda: (1.0 + 0.3 * n) / max(1, shape[-1]),
                 "forget": lambda: 3.0 + 3.0 * u,                                                  # gates near one, as trained ones are
                 "rate": lambda: torch.log(1.0 + 3.0 * u),                                         # decays between e^-0.001 and e^-0.4 a token
                 "pace": lambda: torch.log(torch.expm1(torch.exp(math.log(0.001) + u * math.log(100.0))))}[how]().to(torch.bfloat16)
        out[name] = t if how == "table" else t.to(dtype)
    return out


def lengths_of(case):
    """Cached tokens (decode, mixed) or prompt lengths of the requests: spread evenly between the shortest and the longest, out of order."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    spread = [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)] if n > 1 else [hi]
    return [spread[(7 * i) % n] if n % 7 else spread[(5 * i) % n] if n % 5 else spread[i] for i in range(n)]


def tokens_of(case, seed):
    """Per request: the ids it brings, cached ones first; for "mixed" one more request, the portion."""
    g = torch.Generator().manual_seed(2 * int(seed))
    vocab = VOCAB_QWEN if case["family"] == "qwen" else VOCAB_DESIGN
    more = {"decode": 1, "mixed": 1, "prompt": 0, "whole": case.get("steps", 0)}[case["kind"]]
    sizes = [n + more for n in lengths_of(case)] + ([case["portion"]] if case["kind"] == "mixed" else [])
    return [torch.randint(0, vocab, (n,), generator=g).tolist() for n in sizes]


def wanted(n):
    """Places of a prompt of n tokens whose logits are asked for: the last, as a server wants it, and seven before it, as scoring does."""
    return sorted({(n * (i + 1)) // 8 - 1 for i in range(8) if (n * (i + 1)) // 8 > 0})


# ---- what a program has in hand, and one pass -------------------------------------------------------------------------
def prepare(case, seed):
    from spyinfer_amd.config.registry import architecture_of
    from spyinfer_amd.engine.batch import StepEntry
    from spyinfer_amd.engine.runner import ModelRunner, bind_weights

    raw = config_of(case)
    arch = architecture_of(raw)
    model = arch.build(arch.config_cls.from_dict(raw))
    bind_weights(model, tensors_of(case, seed), torch.device(DEVICE), "both")
    tokens = tokens_of(case, seed)
    pages = sum(-(-(len(t) + 1) // PAGE) for t in tokens) + 8
    runner = ModelRunner(model, case["dtype"], DEVICE, PAGE, pages, max(8, len(tokens)), MOST_TOKENS, enforce_eager=False, max_model_len=MODEL_LEN)
    state = dict(kind=case["kind"], runner=runner, tokens=tokens, lengths=lengths_of(case), entry=StepEntry, live=[], steps=case.get("steps", 0))
    if case["kind"] in ("decode", "mixed"):
        # the requests' contexts come from the model itself, in steps of at most the engine's budget
        waiting, room = [], 0
        for i, n in enumerate(state["lengths"] + [None]):
            if n is None or room + n > MOST_TOKENS:
                runner.step(waiting)
                waiting, room = [], 0
            if n is not None:
                rc = runner.manager.admit("r%d" % i)
                runner.manager.reserve(rc, n)
                waiting.append(StepEntry(rc, tokens[i][:n]))
                state["live"].append(rc)
                room += n
    # a program that serves has run steps of this kind before
    for _ in range(2):
        run(state)
    return state


def run(state):
    runner, tokens, Entry = state["runner"], state["tokens"], state["entry"]
    manager = runner.manager
    if state["kind"] in ("decode", "mixed"):
        entries = []
        for rc, t in zip(state["live"], tokens):
            manager.reserve(rc, 1)
            entries.append(Entry(rc, t[-1:], (0,)))
        new = None
        if state["kind"] == "mixed":
            new = manager.admit("new")
            manager.reserve(new, len(tokens[-1]))
            entries.append(Entry(new, tokens[-1], (len(tokens[-1]) - 1,)))
        logits = runner.step(entries)
        for rc, n in zip(state["live"], state["lengths"]):
            if not manager.rewind(rc, n):
                raise RuntimeError("the step cannot be taken back")
        if new is not None:
            manager.release(new)
        return logits
    live = [manager.admit("r%d" % i) for i in range(len(tokens))]
    entries = []
    for rc, t, n in zip(live, tokens, state["lengths"]):
        manager.reserve(rc, n)
        entries.append(Entry(rc, t[:n], wanted(n) if state["kind"] == "prompt" else (n - 1,)))
    out = [runner.step(entries)]
    for s in range(state["steps"]):
        if s == 0:
            out[0] = out[0].clone()         # a step's logits are good until the next step
        entries = []
        for rc, t, n in zip(live, tokens, state["lengths"]):
            manager.reserve(rc, 1)
            entries.append(Entry(rc, t[n + s:n + s + 1], (0,)))
        out.append(runner.step(entries).clone())
    for rc in live:
        manager.release(rc)
    return out


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def work(case):
    cfg, size = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    lengths = lengths_of(case)
    # (tokens run, keys before them) of every entry of every step; rows of logits; steps
    if case["kind"] == "decode":
        steps, rows = [[(1, n) for n in lengths]], len(lengths)
    elif case["kind"] == "mixed":
        steps, rows = [[(1, n) for n in lengths] + [(case["portion"], 0)]], len(lengths) + 1
    elif case["kind"] == "prompt":
        steps, rows = [[(n, 0) for n in lengths]], sum(len(wanted(n)) for n in lengths)
    else:
        steps = [[(n, 0) for n in lengths]] + [[(1, n + s) for n in lengths] for s in range(case["steps"])]
        rows = len(lengths) * len(steps)
    vocab = VOCAB_QWEN if case["family"] == "qwen" else VOCAB_DESIGN
    flops, moved = 2.0 * rows * vocab * case["width"], 4.0 * rows * vocab
    for step in steps:
        T = sum(t for t, _ in step)
        moved += size * (vocab * case["width"] + T * case["width"])
        for name, shape, how in tensor_list(case):
            if how not in ("matrix", "out") or len(shape) != 2 or name in ("embed", "head", "bigram", "model.embed_tokens.weight", "lm_head.weight"):
                continue
            n = shape[0] * shape[1]
            if ".mlp.e" in name:                     # of 32 experts a token uses four: their rows, and the experts that T tokens touch
                flops += 2.0 * n * T * 4 / 32
                moved += size * n * (1.0 - (1.0 - 4 / 32) ** T)
            else:
                flops += 2.0 * n * T
                moved += size * n
        for i in range(case["layers"]):
            layer = cfg["layers"][i] if "layers" in cfg else None
            m = layer["mixer"] if layer else dict(heads=cfg["num_attention_heads"], kv_heads=8, dim=128, vdim=128)
            kind = layer["type"] if layer else "attention"
            for t, before in step:
                if kind in ("attention", "latent_attention"):
                    reach = (m.get("mask") or {}).get("size") or 1 << 30
                    seen = [min(before + j + 1, reach) for j in ((0, t - 1) if t > 1 else (0,))]
                    pairs = t * (seen[0] + seen[-1]) / 2
                    if kind == "attention":
                        flops += 2.0 * pairs * m["heads"] * (m["dim"] + m["vdim"])
                        moved += size * (min(before, reach) + t) * m["kv_heads"] * (m["dim"] + m["vdim"])
                    else:
                        flops += 2.0 * pairs * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
                        moved += size * (min(before, reach) + t) * (m["kv_rank"] + m["rot_dim"])
                elif kind == "mingru":
                    flops += 8.0 * t * m["width"]
                    moved += 4.0 * 2 * m["width"]
                else:
                    flops += (4.0 if kind == "mlstm" else 8.0) * t * m["heads"] * m["dim"] * m["vdim"]
                    moved += 4.0 * 2 * m["heads"] * m["dim"] * m["vdim"]
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # four times the distance from 64 bits that the listed and a dozen drawn cases had: up to 1.3e-6 in float32, 0.0071 in bfloat16
    if case["dtype"] == "float32":
        return {"rel": 6e-6, "max": 1e-4}
    return {"rel": 0.028, "max": 0.2}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] in ("decode", "mixed") and sum(lengths_of(case)) * case["width"] ** 2 * case["layers"] > 2.2e13:
        return None
    w, tokens = tensors_of(case, seed), tokens_of(case, seed)
    places = []                                    # rows of the flat batch whose logits are wanted, step by step
    starts = [0]
    for t in tokens:
        starts.append(starts[-1] + len(t))
    lengths = lengths_of(case)
    if case["kind"] == "prompt":
        places = [[starts[r] + p for r, n in enumerate(lengths) for p in wanted(n)]]
    elif case["kind"] == "whole":
        places = [[starts[r] + n - 1 + s for r, n in enumerate(lengths)] for s in range(case["steps"] + 1)]
    else:
        places = [[starts[r + 1] - 1 for r in range(len(tokens))]]
    flat = [p for step in places for p in step]
    with torch.no_grad():
        x, head = FORWARD[case["family"]](config_of(case), w, tokens, flat)
        logits = torch.cat([x @ head[r:r + 16384].double().T for r in range(0, head.shape[0], 16384)], dim=1)
    if case["kind"] in ("decode", "mixed"):
        return logits
    out, at = [], 0
    for step in places:
        out.append(logits[at:at + len(step)])
        at += len(step)
    return out


def rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def mul(x, w):
    return x @ w.double().T


def silu(z):
    return z * torch.sigmoid(z)


def turned(x, freq, dims, mag=1.0):
    """The first ``dims`` entries of every head of x [T, heads, n] rotated by the position, pair (i, i + dims / 2)."""
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * freq[None, :]
    c, s = (torch.cos(ang) * mag)[:, None, :], (torch.sin(ang) * mag)[:, None, :]
    a, b = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., dims:]], dim=-1)


def frequencies(dims, base):
    return float(base) ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) / dims)


def attend(q, k, v, scale, window=None, chunk=None, sink=None):
    """One sequence: q [T, H, d], k and v [T, G, ..]; a group of query heads at a time."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    pos = torch.arange(T, device=q.device)
    hidden = pos[None, :] > pos[:, None]
    if window:
        hidden = hidden | (pos[None, :] <= pos[:, None] - window)
    if chunk:
        hidden = hidden | (pos[None, :] // chunk != pos[:, None] // chunk)
    out = []
    for g in range(G):
        s = (q[:, g * (H // G):(g + 1) * (H // G)].permute(1, 0, 2).contiguous() @ k[:, g].T.contiguous()) * scale
        s.masked_fill_(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[g * (H // G):(g + 1) * (H // G), None, None].expand(-1, T, 1)], dim=-1)
        p = torch.softmax(s, dim=-1)[..., :T]
        out.append((p @ v[:, g].contiguous()).permute(1, 0, 2))
    return torch.cat(out, dim=1)


def each(tokens, f):
    """f on every sequence's part of a flat batch, put together again."""
    out, at = [], 0
    for t in tokens:
        out.append(f(slice(at, at + len(t))))
        at += len(t)
    return torch.cat(out)


def ids_of(tokens):
    return torch.tensor([i for t in tokens for i in t], device=DEVICE)


def qwen(cfg, w, tokens, rows):
    eps, H = cfg["rms_norm_eps"], cfg["num_attention_heads"]
    freq = frequencies(128, cfg["rope_theta"])
    x = w["model.embed_tokens.weight"][ids_of(tokens)].double()
    for i in range(cfg["num_hidden_layers"]):
        p = lambda n: w["model.layers.%d.%s.weight" % (i, n)]
        h = rms(x, eps, p("input_layernorm"))
        q, k, v = (mul(h, p("self_attn.%s_proj" % n)).view(len(h), -1, 128) for n in "qkv")
        q, k = rms(q, eps, p("self_attn.q_norm")), rms(k, eps, p("self_attn.k_norm"))
        a = each(tokens, lambda s: attend(turned(q[s], freq, 128), turned(k[s], freq, 128), v[s], 128 ** -0.5))
        x = x + mul(a.reshape(len(h), H * 128), p("self_attn.o_proj"))
        h = rms(x, eps, p("post_attention_layernorm"))
        x = x + mul(silu(mul(h, p("mlp.gate_proj"))) * mul(h, p("mlp.up_proj")), p("mlp.down_proj"))
    return rms(x[rows], eps, w["model.norm.weight"]), w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]


def balelorn(cfg, w, tokens, rows):
    eps, ids, first = cfg["norm"]["eps"], ids_of(tokens), None
    x = rms(w["embed"][ids].double(), eps, w["embed.norm"])
    for i, layer in enumerate(cfg["layers"]):
        p = lambda n: w["l%d.%s" % (i, n)]
        m, T = layer["mixer"], len(x)
        h = rms(x, eps, p("norm1"))
        q, k, own = (mul(h, p("mix." + n)).view(T, -1, 128) for n in "qkv")
        lam = p("mix.vmix").double()
        v = own if first is None else (1.0 - lam) * own + lam * first
        first = own if first is None else first
        freq, chunk = frequencies(m["rot"]["dims"], m["rot"]["base"]), m["mask"]["size"] if m["mask"] else None
        a = each(tokens, lambda s: attend(turned(q[s], freq, 64), turned(k[s], freq, 64), v[s], m["scale"], chunk=chunk, sink=p("mix.sink").double()))
        y = mul(a.reshape(T, -1) * torch.sigmoid(mul(h, p("mix.g"))), p("mix.o"))
        x = x + rms(y, eps, p("norm1b")) * p("ls1").double()
        h = rms(x, eps, p("norm2"))
        if layer["mlp"]["kind"] == "dense":
            z = mul(h, p("mlp.gate"))
            y = mul(0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3))) * mul(h, p("mlp.up")), p("mlp.down"))
        else:
            chosen, y, limit = p("mlp.table")[ids], torch.zeros_like(h), layer["mlp"]["expert"]["limit"]
            for e in range(layer["mlp"]["router"]["experts"]):
                at = (chosen == e).any(dim=-1).nonzero()[:, 0]
                g = mul(h[at], p("mlp.e%d.gate" % e)).clamp(max=limit)
                u = mul(h[at], p("mlp.e%d.up" % e)).clamp(min=-limit, max=limit)
                y[at] += mul(g * torch.sigmoid(1.702 * g) * (u + 1.0), p("mlp.e%d.down" % e)) / chosen.shape[1]
        x = x + rms(y, eps, p("norm2b")) * p("ls2").double()
    return rms(x[rows], eps, w["final.norm"]), w["head"]


def conv_silu(x, taps):
    n = taps.shape[1]
    pad = torch.cat([torch.zeros((n - 1, x.shape[1]), dtype=x.dtype, device=x.device), x])
    return silu(sum(pad[j:j + len(x)] * taps[:, j].double() for j in range(n)))


def unit(x):
    return x / torch.sqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6)


def matrix_memory(q, k, v, ig, fg):
    """One sequence: q, k [T, H, d], v [T, H, dv], log gates [T, H]."""
    S, n, mx = k.new_zeros(k.shape[1], k.shape[2], v.shape[2]), k.new_zeros(k.shape[1:]), k.new_zeros(k.shape[1])
    out = torch.empty_like(v)
    for t in range(len(q)):
        new = torch.maximum(fg[t] + mx, ig[t])
        a, b = torch.exp(fg[t] + mx - new), torch.exp(ig[t] - new)
        bk = b[:, None] * k[t]
        S = a[:, None, None] * S + bk[:, :, None] * v[t][:, None, :]
        n = a[:, None] * n + bk
        mx = new
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-mx)) + 1e-6
        out[t] = (q[t][:, None, :] @ S)[:, 0] / den[:, None]
    return out


def delta_rule(q, k, v, beta, decay):
    """One sequence: q, k, decay [T, H, d], v [T, H, dv], beta [T, H]."""
    S, out = k.new_zeros(k.shape[1], k.shape[2], v.shape[2]), torch.empty_like(v)
    for t in range(len(q)):
        S = decay[t][:, :, None] * S
        u = beta[t][:, None] * (v[t] - (k[t][:, None, :] @ S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None, :]
        out[t] = (q[t][:, None, :] @ S)[:, 0]
    return out


def sodedra(cfg, w, tokens, rows):
    eps = cfg["norm"]["eps"]
    x = w["embed"][ids_of(tokens)].double()
    for i, layer in enumerate(cfg["layers"]):
        p = lambda n: w["l%d.%s" % (i, n)]
        m, T = layer["mixer"], len(x)
        h = rms(x, eps) * (1.0 + p("norm1").double())
        of = lambda n: mul(h, p("mix." + n))
        if layer["type"] == "attention":
            q, k, v = ((of(n) + p("mix.%s.b" % n).double()).view(T, -1, 128) for n in "qkv")
            r = m["rot"]["scaling"]
            f = frequencies(64, m["rot"]["base"])
            turns = r["original"] * f / (2.0 * math.pi)            # of the original context
            s = ((turns - r["low"]) / (r["high"] - r["low"])).clamp(0.0, 1.0)
            f = (1.0 - s) * f / r["factor"] + s * f
            a = each(tokens, lambda c: attend(turned(q[c], f, 64), turned(k[c], f, 64), v[c], m["scale"], window=m["mask"]["size"]))
            y = mul(a.reshape(T, -1) * torch.sigmoid(of("g")), p("mix.o"))
        elif layer["type"] == "mlstm":
            H, cap = m["heads"], m["gate_cap"]
            q, k, v = of("q").view(T, H, -1) * m["dim"] ** -0.5, of("k").view(T, H, -1), of("v").view(T, H, -1)
            ig = cap * torch.tanh((of("i") + p("mix.i.b").double()) / cap)
            fg = torch.nn.functional.logsigmoid(cap * torch.tanh((of("f") + p("mix.f.b").double()) / cap))
            o = each(tokens, lambda c: matrix_memory(q[c], k[c], v[c], ig[c], fg[c]))
            y = mul(rms(o, eps).reshape(T, -1) * p("mix.norm").double() * torch.sigmoid(of("g")), p("mix.o"))
        else:
            H, G, d = m["heads"], m["kv_heads"], m["dim"]
            q, k, v = (each(tokens, lambda c: conv_silu(mul(h[c], p("mix." + n)), p("mix.%s.conv" % n))) for n in "qkv")
            q, k = unit(q.view(T, G, d)) * d ** -0.5, unit(k.view(T, G, d))
            q, k, v = q.repeat_interleave(H // G, dim=1), k.repeat_interleave(H // G, dim=1), v.view(T, H, -1)
            dt = torch.nn.functional.softplus(mul(of("a1"), p("mix.a2")) + p("mix.dt_bias").double()).view(T, H, d)
            decay = torch.exp(-torch.exp(p("mix.A_log").double())[None, :, None] * dt)
            beta = torch.sigmoid(of("b"))
            o = each(tokens, lambda c: delta_rule(q[c], k[c], v[c], beta[c], decay[c]))
            y = mul((rms(o, eps, p("mix.norm")) * torch.sigmoid(mul(of("g1"), p("mix.g2"))).view(T, H, -1)).reshape(T, -1), p("mix.o"))
        x = x + y + mul(silu(mul(h, p("mlp.gate"))) * mul(h, p("mlp.up")), p("mlp.down"))
    return rms(x[rows], eps) * (1.0 + w["final.norm"].double()), w["embed"]


def sefevik(cfg, w, tokens, rows):
    eps, bg = cfg["norm"]["eps"], cfg["embedding"]["bigram"]
    pair = [bg["buckets"] if j == 0 else (t[j - 1] * bg["mul_prev"] + t[j] * bg["mul_cur"]) % bg["buckets"] for t in tokens for j in range(len(t))]
    x = w["embed"][ids_of(tokens)].double() + w["bigram"][torch.tensor(pair, device=DEVICE)].double()
    results, kept = [x], {}
    for i, layer in enumerate(cfg["layers"]):
        p = lambda n: w["l%d.%s" % (i, n)]
        m, T = layer["mixer"], len(x)
        if layer["type"] == "mingru":
            z, u = torch.sigmoid(mul(x, p("mix.z")) + p("mix.z.b").double()), mul(x, p("mix.x")) + p("mix.x.b").double()
            c = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))

            def walk(s):
                state, out = c.new_zeros(c.shape[1]), torch.empty_like(c[s])
                for t in range(len(out)):
                    state = (1.0 - z[s][t]) * state + z[s][t] * c[s][t]
                    out[t] = state
                return out
            y = mul(each(tokens, walk) * silu(mul(x, p("mix.g"))), p("mix.o"))
        else:
            H, r, rot = m["heads"], m["kv_rank"], m["rot"]
            sc, f = rot["scaling"], frequencies(64, rot["base"])
            edge = lambda turns: 64 * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
            lo, hi = max(math.floor(edge(sc["fast"])), 0), min(math.ceil(edge(sc["slow"])), 63)
            ramp = ((torch.arange(32, dtype=torch.float64, device=DEVICE) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
            f, mag = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
            if "kv_from" not in m:
                d = mul(x, p("mix.dkv"))
                kept[i] = (rms(d[:, :r], eps, p("mix.dkv.norm")), each(tokens, lambda s: turned(d[s, None, r:], f, 64, mag)))
            c, kr = kept[m.get("kv_from", i)]
            q = mul(x, p("mix.q")).view(T, H, 192)
            k, v = torch.cat([mul(c, p("mix.uk")).view(T, H, 128), kr.expand(T, H, 64)], dim=-1), mul(c, p("mix.uv")).view(T, H, 128)
            a = each(tokens, lambda s: attend(torch.cat([q[s, :, :128], turned(q[s, :, 128:], f, 64, mag)], dim=-1), k[s], v[s], m["scale"],
                                              window=m["mask"]["size"], sink=p("mix.sink").double()))
            y = mul(a.reshape(T, -1), p("mix.o"))
        x = x + rms(y, eps, p("norm1"))
        act = torch.nn.functional.softplus(p("mlp.act").double())
        z = mul(x, p("mlp.up"))
        z = torch.where(z > 0, act[0] * z * z + 0.5 * z, (0.5 + act[1]) * (torch.expm1(z.clamp(max=0.0)) - z) + 0.5 * z)
        x = x + rms(mul(z, p("mlp.down")), eps, p("norm2"))
        results.append(x)
        x = sum(a * r for a, r in zip(p("dwa").double(), results))
    return rms(x[rows], eps, w["final.norm"]), w["head"]


FORWARD = {"qwen": qwen, "balelorn": balelorn, "sodedra": sodedra, "sefevik": sefevik}
