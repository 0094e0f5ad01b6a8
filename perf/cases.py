"""What the engine is measured on: steps and whole answers through its public entry points (`Engine.step`, the
sampler), at the layer sizes that the benchmark names, over the range of batches and lengths that serving brings.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what a program holds before the call: an engine with its weights, requests whose earlier
                        tokens lie in the cache, the tokens of the step
    run(state)          one pass
    work(case)          bytes and flops that a pass cannot do without
    tolerance(case)     how far two correct implementations of the same precision may differ
    exact(case, seed)   the same outputs in 64 bits from the equations, whole sequences, no cache

Five kinds of pass:
    decode   one step in which every request brings one token behind its context (a step of a chat service at rest)
    prompt   one step with whole prompts (the time to the first token)
    portion  one step with the next portion of a prompt behind what is cached (long documents in portions), beside
             requests that decode (continuous batching)
    answer   prompts, then a token a request and step, then the requests end (a whole batch from start to end)
    sample   the choice of the next tokens from a step's logits
A step of `decode` and `portion` is taken back afterwards (the requests' last tokens are forgotten, their pages
stay), so that every pass is the same step; models whose layers keep a state that moves on run whole answers instead.
The tokens of a step are given, not fed back, so that outputs of two implementations can be compared.
"""
import hashlib
import math
import random

import torch

from litinfer_amd import benchmark
from litinfer_amd.engine import Engine, StepEntry
from litinfer_amd.sampling import Sampler, SamplingParams

PAGE = 16
DTYPES = {"bf16": ("bfloat16", torch.bfloat16), "fp32": ("float32", torch.float32)}
PORTION = 2048                              # tokens a step while contexts are laid down
EXACT_FLOPS = 5.0e14                        # what 64-bit arithmetic does in some ten seconds here


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest step there is: one chat on the smallest member of the family; launches and latency
        dict(name="decode_one_0p5b", kind="decode", model="qwen2", size="0.5b", layers=24, dtype="bf16", requests=1, shortest=300, longest=300),
        # the benchmark's headline: eight requests at the 7B sizes, contexts up to 4,096
        dict(name="decode_8_7b", kind="decode", model="qwen2", size="7b", layers=28, dtype="bf16", requests=8, shortest=2047, longest=4090),
        # a full batch of a small model with contexts of all lengths
        dict(name="decode_64_1p5b", kind="decode", model="qwen2", size="1.5b", layers=28, dtype="bf16", requests=64, shortest=100, longest=2001),
        # the benchmark's prompt
        dict(name="prompt_2048_7b", kind="prompt", model="qwen2", size="7b", layers=28, dtype="bf16", requests=1, shortest=2048, longest=2048),
        # continuous batching: a portion of one prompt beside decoding requests, an odd number of rows
        dict(name="mixed_1p5b", kind="portion", model="qwen2", size="1.5b", layers=28, dtype="bf16", cached=517, tokens=990, requests=37, shortest=50, longest=1500),
        # a long document at the 32B layer sizes (8 of its layers), a late portion
        dict(name="portion_32b_behind_16000", kind="portion", model="qwen2", size="32b", layers=8, dtype="bf16", cached=16000, tokens=1999, requests=0, shortest=0, longest=0),
        # the 32-bit path: short answers
        dict(name="answer_fp32_1p5b", kind="answer", model="qwen2", size="1.5b", layers=28, dtype="fp32", requests=3, shortest=40, longest=500, steps=8),
        # state-space layers, differential attention, routed experts: one long prompt and its answer's beginning
        dict(name="answer_sogenex", kind="answer", model="sogenex", size="1.5b", layers=6, dtype="bf16", requests=1, shortest=2048, longest=2048, steps=16),
        # delta rule, retention, routed experts: a batch of prompts of all lengths
        dict(name="answer_kufolorn", kind="answer", model="kufolorn", size="1.5b", layers=6, dtype="bf16", requests=8, shortest=20, longest=481, steps=16),
        # residual streams, latent attention, channel-wise delta rule: two prompts longer than the window
        dict(name="answer_dimelix", kind="answer", model="dimelix", size="1.5b", layers=6, dtype="bf16", requests=2, shortest=1100, longest=1501, steps=16),
        # lightning, chunked and latent attention, routed experts: many short chats
        dict(name="answer_besorax", kind="answer", model="besorax", size="1.5b", layers=6, dtype="bf16", requests=32, shortest=9, longest=131, steps=16),
        # the choice of tokens for a full batch: greedy, temperature, top-k with top-p
        dict(name="sample_64", kind="sample", rows=64, vocab=151936),
    ]


def _spread(rng, low, high):
    """A whole number between the two, evenly over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "portion", "portion", "answer", "answer", "answer", "sample"])
    if kind == "sample":
        return dict(kind=kind, rows=_spread(rng, 1, 128), vocab=rng.choice([32000, 151936, 152064]))
    if kind == "decode":
        size = rng.choice(["0.5b", "1.5b", "7b"])
        n = _spread(rng, 1, 64)
        top = min(4090, (24000 if size == "7b" else 65000) // n)
        longest = _spread(rng, 16, top)
        return dict(kind=kind, model="qwen2", size=size, layers=benchmark.SHAPES[size]["num_hidden_layers"], dtype="bf16",
                    requests=n, shortest=max(1, longest // rng.choice([1, 2, 8])), longest=longest)
    if kind == "prompt":
        size = rng.choice(["0.5b", "1.5b", "7b"])
        n = _spread(rng, 1, 8)
        longest = _spread(rng, 8, (2048 if size == "7b" else 4096) // n)
        return dict(kind=kind, model="qwen2", size=size, layers=benchmark.SHAPES[size]["num_hidden_layers"], dtype="bf16",
                    requests=n, shortest=max(2, longest // rng.choice([1, 2, 4])), longest=longest)
    if kind == "portion":
        if rng.random() < 0.4:
            return dict(kind=kind, model="qwen2", size="32b", layers=8, dtype="bf16", cached=_spread(rng, 500, 16000),
                        tokens=_spread(rng, 32, 2000), requests=0, shortest=0, longest=0)
        longest = _spread(rng, 16, 2000)
        return dict(kind=kind, model="qwen2", size="1.5b", layers=28, dtype="bf16", cached=_spread(rng, 1, 4000),
                    tokens=_spread(rng, 16, 2000), requests=_spread(rng, 1, 48), shortest=max(1, longest // 4), longest=longest)
    model = rng.choice(["qwen2", "sogenex", "kufolorn", "dimelix", "besorax"])
    n = _spread(rng, 1, 4 if model == "qwen2" else 32)
    longest = _spread(rng, 4, min(2048, (1024 if model == "qwen2" else 2560) // n))
    return dict(kind="answer", model=model, size="1.5b", layers=28 if model == "qwen2" else 6, dtype="fp32" if model == "qwen2" else "bf16",
                requests=n, shortest=max(2, longest // rng.choice([1, 2, 8])), longest=longest, steps=rng.randint(2, 16))


def lengths(case):
    """The requests' lengths, spread evenly from the shortest to the longest, in an order that mixes them."""
    n, low, high = case["requests"], case["shortest"], case["longest"]
    out = [low + (high - low) * i // max(1, n - 1) if n > 1 else high for i in range(n)]
    random.Random(7).shuffle(out)
    return out


def sequences(case):
    """[(tokens laid down before the step, tokens of the step)] of the requests of a `decode` or `portion` case."""
    seqs = [(n, 1) for n in lengths(case)]
    return [(case["cached"], case["tokens"])] + seqs if case["kind"] == "portion" else seqs


def config(case):
    if case["model"] == "qwen2":
        return dict(benchmark.SHAPES[case["size"]], num_hidden_layers=case["layers"], max_position_embeddings=32768)
    return getattr(benchmark, case["model"] + "_config")(case["size"], case["layers"])


def vocabulary(cfg):
    return cfg["vocab_size"] if "vocab_size" in cfg else cfg["vocab"]


# --------------------------------------------------------------------------------------------------------- weights
def tensors(cfg):
    """Name -> (shape, how it is drawn) of every tensor that a checkpoint of this model holds."""
    t = {}

    def ff(p, width, inner, names):
        for n in names:
            t[p + n] = ((width, inner) if n == "down" else (inner, width), "normal")

    if "architecture" not in cfg:
        W, H, G, D, F = (cfg[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size"))
        t["model.embed_tokens.weight"] = ((cfg["vocab_size"], W), "normal")
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            for n in ("input_layernorm", "post_attention_layernorm"):
                t[f"{p}{n}.weight"] = ((W,), "one_plus_normal")
            for n, rows in (("q", H), ("k", G), ("v", G)):
                t[f"{p}self_attn.{n}_proj.weight"] = ((rows * D, W), "normal")
                t[f"{p}self_attn.{n}_proj.bias"] = ((rows * D,), "normal")
            t[f"{p}self_attn.o_proj.weight"] = ((W, H * D), "normal")
            for n in ("gate", "up"):
                t[f"{p}mlp.{n}_proj.weight"] = ((F, W), "normal")
            t[f"{p}mlp.down_proj.weight"] = ((W, F), "normal")
        t["model.norm.weight"] = ((W,), "one_plus_normal")
        if not cfg["tie_word_embeddings"]:
            t["lm_head.weight"] = ((cfg["vocab_size"], W), "normal")
        return t
    kind, W = cfg["architecture"], cfg["width"]
    t["embed"] = ((cfg["vocab"], W), "normal")
    plain = {"Sogenex": "normal", "Kufolorn": "normal", "Dimelix": "normal", "Besorax": "one_plus_normal"}[kind]

    def norm(name):
        t[name] = ((W,), plain)
        if kind == "Besorax":
            t[name + ".alpha"], t[name + ".b"] = ((), "one_plus_normal"), ((W,), "normal")

    def mixer(p, what, m):
        if what == "parallel":
            mixer(p + "left.", "distance" if kind == "Dimelix" else "attention", m["left"])
            mixer(p + "right.", "channel_delta" if kind == "Dimelix" else "retention", m["right"])
            return
        H, D = m["heads"], m.get("dim", 0)
        V, G = m.get("vdim", D), m.get("kv_heads", H)
        mats = {"o": (W, H * V)}
        if what == "mamba2":
            inner, bc = H * V, 2 * m["groups"] * m["state"]
            mats["in"] = (2 * inner + bc + H, W)
            t[p + "conv"], t[p + "conv.b"] = ((inner + bc, m["conv"]), "normal"), ((inner + bc,), "zeros")
            t[p + "dt_bias"], t[p + "A_log"], t[p + "D"] = ((H,), "normal"), ((H,), "normal"), ((H,), "ones")
            t[p + "norm"] = ((inner,), "one_plus_normal")
        elif what == "delta":
            mats.update(g=(H * V, W), b=(H, W), a=(H, W), q=(G * D, W), k=(G * D, W), v=(H * V, W))
            for n, rows in (("q", G * D), ("k", G * D), ("v", H * V)):
                t[f"{p}{n}.conv"] = ((rows, m["conv"]), "normal")
            t[p + "A_log"], t[p + "dt_bias"], t[p + "norm"] = ((H,), "normal"), ((H,), "normal"), ((V,), "one_plus_normal")
        elif what == "retention":
            mats.update(q=(H * D, W), k=(H * D, W), v=(H * V, W), g=(H * V, W))
        elif what == "lightning":
            mats.update(q=(H * D, W), k=(H * D, W), v=(H * V, W), g=(H * V, W))
            t[p + "norm"] = ((H * V,), "one_plus_normal")
        elif what == "channel_delta":
            low = 64
            mats.update(r=(H * D, W), k=(H * D, W), v=(H * D, W), g=(H * D, W), a=(H * D, W), w1=(low, W), w2=(H * D, low))
            for n in ("a.b", "w0"):
                t[p + n] = ((H * D,), "normal")
            t[p + "norm"] = ((H * D,), "one_plus_normal")
        elif what == "latent_attention":
            R = m.get("rot_dim", 0)
            mats.update(dkv=(m["kv_rank"] + R, W), uk=(H * D, m["kv_rank"]), uv=(H * V, m["kv_rank"]))
            t[p + "dkv.norm"] = ((m["kv_rank"],), "one_plus_normal")
            if "q_rank" in m:
                mats.update(dq=(m["q_rank"], W), uq=(H * (D + R), m["q_rank"]))
                t[p + "dq.norm"] = ((m["q_rank"],), "one_plus_normal")
            else:
                mats["q"] = (H * (D + R), W)
        else:                                                   # attention, distance
            two = 2 if "diff" in m else 1
            mats.update(q=(H * two * D, W))
            if m.get("kv_from") is None:
                mats.update(k=(G * two * D, W))
                if what != "distance":
                    mats.update(v=(G * V, W))
            if "diff" in m:
                for n in ("lq1", "lk1", "lq2", "lk2"):
                    t[p + n] = ((D,), "normal")
            if kind == "Kufolorn":
                mats["g"] = (H, W)
                for n, rows in (("q", H), ("k", G), ("v", G)):
                    t[f"{p}{n}.b"] = ((rows * D,), "normal")
                for n, rows in (("q", H), ("k", G)):
                    t[f"{p}{n}.norm"] = ((rows * D,), "one_plus_normal")
            if kind == "Dimelix":
                for n in ("q", "k"):
                    t[f"{p}{n}.norm"] = ((D,), "one_plus_normal")
            if kind in ("Kufolorn", "Besorax") or (kind == "Dimelix" and what == "attention"):
                t[p + "sink"] = ((H,), "normal")
        if kind == "Dimelix" and what != "channel_delta":
            mats["g"] = (H * V, W)
        if kind == "Besorax" and what == "latent_attention":
            t[p + "sink"] = ((H,), "normal")
        for n, shape in mats.items():
            t[p + n] = (shape, "normal")

    for i, L in enumerate(cfg["layers"]):
        p = f"l{i}."
        norm(p + "norm1")
        norm(p + "norm2")
        mixer(p + "mix.", L["type"], L["mixer"])
        f, q = L["mlp"], p + "mlp."
        if kind == "Dimelix":
            for hc in ("hc1.", "hc2."):
                S = cfg["streams"]
                t[p + hc + "in"], t[p + hc + "out"], t[p + hc + "mix"] = ((S,), "one_plus_normal"), ((S,), "one_plus_normal"), ((S, S), "normal")
            t[q + "act"] = ((2,), "normal")
        gated = ("gate", "up", "down") if kind == "Kufolorn" or (kind == "Besorax" and f["kind"] == "dense") else ("up", "down")
        if f["kind"] == "dense":
            ff(q, W, f["ff"], gated)
        else:
            r = f["router"]
            t[q + "router"] = ((r["experts"] + r.get("identity", 0), W), "normal")
            if kind == "Sogenex":
                t[q + "router.b"] = ((r["experts"],), "zeros")
            if kind == "Kufolorn":
                t[q + "correction"] = ((r["experts"] + r["identity"],), "normal")
            for e in range(r["experts"]):
                ff(f"{q}e{e}.", W, f["expert"]["ff"], gated)
            if f.get("shared"):
                ff(q + "shared.", W, f["shared"]["ff"], ("up", "down"))
                if kind == "Sogenex":
                    t[q + "shared.sg"] = ((1, W), "normal")
    norm("final.norm")
    if kind in ("Sogenex", "Besorax"):
        t["head"] = ((cfg["vocab"], W), "normal")
    return t


def _generator(seed, name, device):
    h = hashlib.sha256(f"{seed}:{name}".encode("utf-8")).digest()
    return torch.Generator(device=device).manual_seed(int.from_bytes(h[:8], "little") & 0x7FFFFFFFFFFFFFFF)


# Routed models: a token's class marks the columns of the experts that it belongs to, as the experts of a trained
# model split the vocabulary among them, and the routers read these columns; with purely random routers every
# tenth token would sit so close between two experts that rounding decides, and outputs could not be compared.
#   (the mark of a chosen column in the embedding, of the others, the routers' weight on it, of the rest)
MARKS = {"Sogenex": (10.0, 0.0, 0.5, 0.005), "Kufolorn": (24.0, 0.0, 0.2, 0.001), "Besorax": (4.0 / 39.0, -4.0 / 39.0, 1.5, 0.005)}


def _classes(cfg, g, device):
    """[vocab, outputs] of zeros and ones: the router outputs that a token belongs to."""
    r = next(L["mlp"]["router"] for L in cfg["layers"] if L["mlp"]["kind"] == "moe")
    n, groups = r["experts"] + r.get("identity", 0), r.get("groups") or {"count": 1, "keep": 1}
    score = torch.rand((cfg["vocab"], n), generator=g, device=device)
    per, each = n // groups["count"], r["top"] // groups["keep"]
    if groups["count"] > 1:                                    # as many in each of the kept groups
        kept = torch.rand((cfg["vocab"], groups["count"]), generator=g, device=device).topk(groups["keep"], dim=1).indices
        inside = torch.zeros((cfg["vocab"], groups["count"]), device=device).scatter_(1, kept, 1.0)
        order = score.view(-1, groups["count"], per).argsort(dim=2, descending=True).argsort(dim=2)
        return ((order < each).float() * inside[:, :, None]).view(-1, n)
    return torch.zeros_like(score).scatter_(1, score.topk(r["top"], dim=1).indices, 1.0)


def weight(cfg, seed, name, spec, stored, device):
    """One tensor of the model, from the seed and its name: N(0, 0.02), around one for norms, as `Engine.from_random`
    draws them, but with the residual stream of a trained model: embeddings of unit size, to which every sublayer
    adds a fraction of that (with embeddings of 0.02 the first sublayers drown them, every rounding is carried
    through all layers, and two correct summation orders end up 4 % apart).  In the routed models the marks above
    and decays that remember; streams that keep what they hold."""
    shape, init = spec
    g = _generator(seed, name, device)
    if init in ("zeros", "ones"):
        return torch.full(shape, float(init == "ones"), device=device, dtype=stored)
    t = torch.randn(shape, generator=g, device=device, dtype=torch.float32) * 0.02
    if init == "one_plus_normal":
        t += 1.0
    kind = cfg.get("architecture", "Qwen2")
    if kind == "Qwen2":
        if name == "model.embed_tokens.weight":
            t *= 50.0
        elif name.endswith(("o_proj.weight", "down_proj.weight")):
            t *= (2 * cfg["num_hidden_layers"]) ** -0.5
    elif kind == "Dimelix":
        if name == "embed":
            t *= 50.0 / cfg["embedding"]["scale"]
        elif name.endswith((".hc1.mix", ".hc2.mix")):
            t += torch.eye(shape[0], device=device)
        elif name.endswith((".hc1.out", ".hc2.out")):
            t *= (2 * len(cfg["layers"])) ** -0.5
        elif name.endswith((".hc1.in", ".hc2.in")):
            t /= cfg["streams"]
    else:
        on, off, reads, rest = MARKS[kind]
        if name == "embed":
            c = _classes(cfg, g, device)
            t[:, :c.shape[1]] = off + (on - off) * c + t[:, :c.shape[1]]
        elif name.endswith("mlp.router"):
            t *= rest / 0.02
            t[:, :shape[0]] += reads * torch.eye(shape[0], device=device)
        elif name.endswith(".dt_bias"):                        # steps of 0.01 to 0.2
            t = torch.expm1(torch.exp(torch.rand(shape, generator=g, device=device) * math.log(20.0)) * 0.01).log()
        elif name.endswith(".A_log"):
            t = (1.0 + 7.0 * torch.rand(shape, generator=g, device=device)).log()
        elif name == "final.norm" and kind == "Kufolorn":      # the head is the embedding: it does not see the marks
            t[:16] = -1.0
    return t.to(stored)


# -------------------------------------------------------------------------------------------------- prepare and run
def token_ids(case, seed, cfg):
    """The whole sequence of every request: what is laid down before, the step's tokens, the answer's."""
    g = torch.Generator().manual_seed(int(seed) * 1000003 + 17)
    if case["kind"] in ("decode", "portion"):
        sizes = [a + b for a, b in sequences(case)]
    else:
        sizes = [n + case.get("steps", 0) for n in lengths(case)]
    return [torch.randint(0, vocabulary(cfg), (n,), generator=g).tolist() for n in sizes]


def sampling(case, seed):
    """A third of the rows greedy, a third at a temperature, a third with top-k and top-p, each with its own stream."""
    kinds = [SamplingParams(), dict(temperature=0.7), dict(temperature=0.8, top_k=50, top_p=0.9)]
    out = []
    for i in range(case["rows"]):
        k = kinds[i % 3]
        out.append(k if isinstance(k, SamplingParams) else SamplingParams(seed=seed * 1000 + i, **k))
    return out


def prepare(case, seed):
    device = "cuda:0"
    if case["kind"] == "sample":
        g = torch.Generator(device=device).manual_seed(int(seed))
        logits = torch.randn((case["rows"], case["vocab"]), generator=g, device=device) * 2.5
        return {"kind": "sample", "sampler": Sampler(device), "logits": logits, "params": sampling(case, seed),
                "counters": list(range(case["rows"])), "out": torch.empty(case["rows"], dtype=torch.int32, device=device), "pending": None}
    cfg, (dtype, stored) = config(case), DTYPES[case["dtype"]]
    ids = token_ids(case, seed, cfg)
    pages = sum(-(-len(s) // PAGE) for s in ids) + 8
    eng = Engine.from_random(cfg, seed, dtype=dtype, device=device, page_size=PAGE, num_pages=pages, max_seqs=len(ids) + 1, page_order_seed=0)
    known = tensors(cfg)
    eng.model.load_params(lambda name: weight(cfg, seed, name, known[name], stored, device) if name in known else None)
    state = {"kind": case["kind"], "engine": eng}
    if case["kind"] in ("decode", "portion"):
        before = [a for a, _ in sequences(case)]
        todo = [(i, o, min(o + PORTION, n)) for i, n in enumerate(before) for o in range(0, n, PORTION)]
        while todo:                                            # the contexts, as many tokens a step as a scheduler would take
            batch, total = [], 0
            while todo and total + todo[0][2] - todo[0][1] <= 2 * PORTION and (not batch or todo[0][0] != batch[-1][0]):
                batch.append(todo.pop(0))
                total += batch[-1][2] - batch[-1][1]
            eng.step([StepEntry(i, ids[i][a:b]) for i, a, b in batch])
        state["entries"] = [StepEntry(i, s[n:], [len(s) - n - 1]) for i, (s, n) in enumerate(zip(ids, before))]
    else:
        n = lengths(case)
        state["entries"] = [StepEntry(i, s[:k], [k - 1]) for i, (s, k) in enumerate(zip(ids, n))]
        state["steps"] = [[StepEntry(i, [s[k + j]], [0]) for i, (s, k) in enumerate(zip(ids, n))] for j in range(case.get("steps", 0))]
    return state


def run(state):
    if state["kind"] == "sample":
        if state["pending"] is not None:
            state["pending"].result()                          # the tokens of the step before, as a serving loop reads them
        state["pending"] = state["sampler"].sample_async(state["logits"], state["params"], state["counters"], out=state["out"])
        return state["out"]
    eng, entries = state["engine"], state["entries"]
    logits = eng.step(entries)
    if state["kind"] in ("decode", "portion"):
        for e in entries:
            eng.cache.rewind(e.rid, len(e.tokens))
        return logits
    out = [logits]
    for step in state["steps"]:
        out.append(eng.step(step).clone())                     # (a recorded step's buffer holds until the next one)
    for e in entries:
        eng.finish(e.rid)
    return out


# ------------------------------------------------------------------------------------------------- work and tolerance
def _layer_order(cfg):
    if "architecture" not in cfg:
        return list(range(cfg["num_hidden_layers"]))
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return list(range(n))
    return list(range(loop["start"])) + loop["times"] * list(range(loop["start"], loop["stop"])) + list(range(loop["stop"], n))


def _layer_work(cfg, i, known, es):
    """(bytes of the matrices that every token uses, flops a token in matrices, bytes of one routed expert, experts,
    experts a token, [(bytes a cached token, flops a visible pair, window)], bytes of state a request) of a layer."""
    p = f"model.layers.{i}." if "architecture" not in cfg else f"l{i}."
    size = sum(math.prod(s) for n, (s, _) in known.items() if n.startswith(p) and len(s) == 2 and ".mlp.e" not in n)
    expert = sum(math.prod(s) for n, (s, _) in known.items() if n.startswith(p + "mlp.e0."))
    if "architecture" not in cfg:
        H, G, D = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        return size * es, 2 * size, 0, 0, 0, [(2 * G * D * es, 4 * H * D, 0)], 0
    L = cfg["layers"][i]
    r = L["mlp"].get("router") or {}
    n, top = r.get("experts", 0), r.get("top", 0)
    used = top * n / max(1, n + r.get("identity", 0))
    pairs, state, extra = [], 0, 0
    ms = [("left", L["mixer"]["left"]), ("right", L["mixer"]["right"])] if L["type"] == "parallel" else [(L["type"], L["mixer"])]
    for what, m in ms:
        H, D = m["heads"], m.get("dim", m.get("state", 0))
        V = m.get("vdim", D)
        if what in ("mamba2", "delta", "lightning", "right"):
            state += H * D * V * 4
            extra += (8 if what in ("delta", "right") else 4) * H * D * V
        elif what == "latent_attention":
            row = m["kv_rank"] + m.get("rot_dim", 0)
            pairs.append((row * es, 2 * H * (D + m.get("rot_dim", 0) + V), 0))
        else:
            G, two = m["kv_heads"], 2 if "diff" in m else 1
            pairs.append(((two * G * D + G * V) * es, 2 * H * two * (D + V), (m.get("mask") or {}).get("size", 0)))
    return size * es, 2 * size + extra + 2 * expert * used, expert * es, n, used, pairs, state


def _step_work(cfg, known, es, segments, wanted):
    """One step: segments of (cached before, new tokens)."""
    T = sum(n for _, n in segments)
    bytes_, flops, W, V = 0.0, 0.0, cfg.get("hidden_size", cfg.get("width")), vocabulary(cfg)
    for i in _layer_order(cfg):
        fixed, a_token, expert, n, used, pairs, state = _layer_work(cfg, i, known, es)
        bytes_ += fixed + expert * (n * (1.0 - (1.0 - used / n) ** T) if n else 0)
        flops += a_token * T
        for start, new in segments:
            bytes_ += 2 * state
            for row, pair, window in pairs:
                seen = start * new + new * (new + 1) / 2.0
                held = start + new
                if window and held > window:
                    seen = sum(min(window, start + j + 1) for j in range(new))
                    held = min(held, window + new)
                bytes_ += row * held
                flops += pair * seen
    return bytes_ + W * V * es + 4.0 * wanted * V + W * es * T, flops + 2.0 * wanted * W * V


def work(case):
    if case["kind"] == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 2.0 * case["rows"] * case["vocab"]}
    cfg = config(case)
    known, es = tensors(cfg), 2 if case["dtype"] == "bf16" else 4
    if case["kind"] in ("decode", "portion"):
        steps = [sequences(case)]
    else:
        n = lengths(case)
        steps = [[(0, k) for k in n]] + [[(k + j, 1) for k in n] for j in range(case.get("steps", 0))]
    each = [_step_work(cfg, known, es, s, len(s)) for s in steps]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    """Whole runs with their sums in another order (prompts in two portions, requests one by one, other tiles) came out
    up to 0.0083 apart in bfloat16 (0.032 of the outputs' size in single values) and 8.5e-7 in float32; four times that."""
    if case["kind"] == "sample":
        return "exact"
    return {"rel": 5e-6, "max": 5e-5} if case["dtype"] == "fp32" else {"rel": 0.03, "max": 0.15}


# ------------------------------------------------------------------------------------------------------ in 64 bits
def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, window=0, chunk=0, sink=None, slopes=None):
    """q [T, H, D], k [T, G, D], v [T, G, V] of one sequence; query i sees j <= i inside its window or chunk."""
    T, H, _ = q.shape
    G = k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=q.dtype, device=q.device)
    at = torch.arange(T, device=q.device)
    for g in range(G):
        hs = slice(g * (H // G), (g + 1) * (H // G))
        kt, vg = k[:, g].t().contiguous(), v[:, g]
        step = max(16, int(2e8 // (T * (H // G))))
        for a in range(0, T, step):
            b = min(T, a + step)
            i, j = at[a:b, None], at[None, :b]
            hidden = j > i
            if window:
                hidden = hidden | (i - j >= window)
            if chunk:
                hidden = hidden | (j // chunk != i // chunk)
            n = b - a
            s = (q[a:b, hs].reshape(-1, q.shape[2]) @ kt[:, :b]).view(n, H // G, b) * scale
            if slopes is not None:
                s = s - slopes[hs][None, :, None] * (i - j)[:, None, :]
            s = s.masked_fill(hidden[:, None, :], -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[hs][None, :, None].expand(n, -1, 1)], dim=2)
            s = torch.softmax(s, dim=2)[:, :, :b]
            out[a:b, hs] = (s.reshape(-1, b) @ vg[:b]).view(n, H // G, -1)
    return out


def _rotate(x, base, dims, halves, factor=1.0):
    """x [T, heads, d]: pairs among the first `dims` columns (a column and the one half behind it, or neighbours)."""
    i = torch.arange(dims // 2, dtype=x.dtype, device=x.device)
    a = torch.arange(x.shape[0], dtype=x.dtype, device=x.device)[:, None] * (base ** (-2.0 * i / dims) / factor)
    c, s = a.cos()[:, None], a.sin()[:, None]
    out = x.clone()
    first, second = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * c - v * s, v * c + u * s
    return out


def _decayed_sum(q, k, v, log_decay):
    """o_i = sum over j <= i of exp(log_decay summed over j+1..i) (q_i . k_j) v_j; q, k [T, H, D], v [T, H, V], log_decay [T, H]."""
    T, H, _ = q.shape
    total = log_decay.cumsum(0)
    later = torch.ones((T, T), dtype=torch.bool, device=q.device).triu(1)
    out = torch.empty_like(v)
    for h in range(H):
        a = (total[:, None, h] - total[None, :, h]).masked_fill(later, -math.inf).exp()
        out[:, h] = ((q[:, h] @ k[:, h].t()) * a) @ v[:, h]
    return out


def _conv(u, w, b=None):
    y = torch.zeros_like(u) if b is None else b.expand_as(u).clone()
    taps = w.shape[1]
    for j in range(taps):
        back = taps - 1 - j
        y[back:] += w[:, j] * u[:u.shape[0] - back]
    return y


def _routed(h, mlp, scores, choice, expert, on_input=False):
    r = mlp["router"]
    groups = r.get("groups")
    if groups and groups["count"] > 1:
        best = choice.view(len(h), groups["count"], -1).amax(2)
        kept = torch.zeros_like(best).scatter_(1, best.topk(groups["keep"], dim=1).indices, 1.0).bool()
        choice = choice.masked_fill(~kept.repeat_interleave(choice.shape[1] // groups["count"], 1), -math.inf)
    idx = choice.topk(r["top"], dim=1).indices
    out = torch.zeros_like(h)
    for e in range(choice.shape[1]):
        rows = (idx == e).any(1).nonzero()[:, 0]
        if len(rows):
            a = scores(idx)[rows][idx[rows] == e][:, None]
            if e >= r["experts"]:
                out[rows] += a * h[rows]
            else:
                out[rows] += expert(e, a * h[rows]) if on_input else a * expert(e, h[rows])
    return out


class _Plain:
    """A model's layers from their equations, in 64 bits, on whole sequences."""

    def __init__(self, cfg, seed, stored, device):
        self.cfg, self.seed, self.stored, self.device = cfg, seed, stored, device
        self.known, self.kind = tensors(cfg), cfg.get("architecture", "Qwen2")
        self.eps = cfg["rms_norm_eps"] if self.kind == "Qwen2" else cfg["norm"]["eps"]
        self.held = {}

    def w(self, name):
        if name not in self.held:
            self.held[name] = weight(self.cfg, self.seed, name, self.known[name], self.stored, self.device).double()
        return self.held[name]

    def lin(self, h, name):
        w = self.w(name)
        return torch.cat([part @ w.t() for part in h.split(4096)])

    def norm(self, x, name):
        if self.kind == "Besorax":
            return torch.tanh(self.w(name + ".alpha") * x) * self.w(name) + self.w(name + ".b")
        return _rms(x, self.eps) * (1.0 + self.w(name))

    def rms(self, x, name):
        return _rms(x, self.eps) * self.w(name)

    # ---- mixers: h holds one sequence
    def attention(self, h, p, m, i):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        V = m.get("vdim", D)
        if "diff" in m:
            q, k, v = self.lin(h, p + "q").view(T, 2 * H, D), self.lin(h, p + "k").view(T, 2 * G, D), self.lin(h, p + "v").view(T, G, V)
            lam = (self.w(p + "lq1") * self.w(p + "lk1")).sum().exp() - (self.w(p + "lq2") * self.w(p + "lk2")).sum().exp() + m["diff"]
            a, b = (_attend(q[:, n::2], k[:, n::2], v, m["scale"], (m.get("mask") or {}).get("size", 0)) for n in (0, 1))
            return self.lin((_rms(a - lam * b, self.eps) * (1.0 - m["diff"])).reshape(T, -1), p + "o")
        if self.kind == "Kufolorn":
            q, k, v = (self.lin(h, p + n) + self.w(p + n + ".b") for n in "qkv")
            rot = m["rot"]
            turn = lambda x: _rotate(x, rot["base"], rot["dims"], True, rot["scaling"]["factor"])  # noqa: E731
            o = _attend(turn(self.rms(q, p + "q.norm").view(T, H, D)), turn(self.rms(k, p + "k.norm").view(T, G, D)), v.view(T, G, V), m["scale"], sink=self.w(p + "sink"))
            return self.lin((o * torch.sigmoid(self.lin(h, p + "g"))[:, :, None]).reshape(T, -1), p + "o")
        if self.kind == "Dimelix":
            q, raw = self.rms(self.lin(h, p + "q").view(T, H, D), p + "q.norm"), self.lin(h, p + "k").view(T, G, D)
            k = self.rms(raw, p + "k.norm")
            if "rot" in m:
                o = _attend(_rotate(q, m["rot"]["base"], m["rot"]["dims"], False), _rotate(k, m["rot"]["base"], m["rot"]["dims"], False),
                            self.lin(h, p + "v").view(T, G, V), m["scale"], sink=self.w(p + "sink"))
            else:
                slopes = torch.tensor([2.0 ** (-8.0 * (n + 1) / H) for n in range(H)], dtype=h.dtype, device=h.device)
                o = _attend(q, k, raw, m["scale"], window=m["mask"]["size"], slopes=slopes)
            return self.lin(o.reshape(T, -1) * torch.sigmoid(self.lin(h, p + "g")), p + "o")
        rot = m["rot"]
        q = _rotate(self.lin(h, p + "q").view(T, H, D), rot["base"], rot["dims"], False)
        if m.get("kv_from") is None:
            self.shared[i] = (_rotate(self.lin(h, p + "k").view(T, G, D), rot["base"], rot["dims"], False), self.lin(h, p + "v").view(T, G, V))
        k, v = self.shared[i if m.get("kv_from") is None else m["kv_from"]]
        return self.lin(_attend(q, k, v, m["scale"], chunk=m["mask"]["size"], sink=self.w(p + "sink")).reshape(T, -1), p + "o")

    def latent_attention(self, h, p, m, i):
        T, H, D, R, V, rank = len(h), m["heads"], m["dim"], m.get("rot_dim", 0), m["vdim"], m["kv_rank"]
        q = (self.lin(self.rms(self.lin(h, p + "dq"), p + "dq.norm"), p + "uq") if "q_rank" in m else self.lin(h, p + "q")).view(T, H, D + R)
        down = self.lin(h, p + "dkv")
        c = self.rms(down[:, :rank], p + "dkv.norm")
        k, v = self.lin(c, p + "uk").view(T, H, D), self.lin(c, p + "uv").view(T, H, V)
        if R:
            q = torch.cat([q[:, :, :D], _rotate(q[:, :, D:], m["rot"]["base"], R, False)], 2)
            k = torch.cat([k, _rotate(down[:, None, rank:], m["rot"]["base"], R, False).expand(T, H, R)], 2)
        o = _attend(q, k, v, m["scale"], sink=self.w(p + "sink") if self.kind == "Besorax" else None).reshape(T, -1)
        if self.kind == "Dimelix":
            o = o * torch.sigmoid(self.lin(h, p + "g"))
        return self.lin(o, p + "o")

    def mamba2(self, h, p, m, i):
        T, H, V, N, G = len(h), m["heads"], m["vdim"], m["state"], m["groups"]
        z, xbc, dt = self.lin(h, p + "in").split([H * V, H * V + 2 * G * N, H], 1)
        xbc = torch.nn.functional.silu(_conv(xbc, self.w(p + "conv"), self.w(p + "conv.b")))
        x, B, C = xbc.split([H * V, G * N, G * N], 1)
        x, B, C = x.view(T, H, V), B.view(T, G, N).repeat_interleave(H // G, 1), C.view(T, G, N).repeat_interleave(H // G, 1)
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"))
        y = _decayed_sum(C, B * dt[:, :, None], x, -self.w(p + "A_log").exp() * dt) + self.w(p + "D")[:, None] * x
        y = y.reshape(T, -1) * torch.nn.functional.silu(z)
        y = _rms(y.view(T, m["norm_groups"], -1), self.eps).reshape(T, -1) * self.w(p + "norm")
        return self.lin(y, p + "o")

    def delta(self, h, p, m, i):
        T, H, G, D, V = len(h), m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        silu = torch.nn.functional.silu
        q, k, v = (silu(_conv(self.lin(h, p + n), self.w(p + n + ".conv"))) for n in "qkv")
        unit = lambda x: x.view(T, G, D) * torch.rsqrt((x.view(T, G, D) ** 2).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k, v = unit(q).repeat_interleave(H // G, 1) * D ** -0.5, unit(k).repeat_interleave(H // G, 1), v.view(T, H, V)
        beta = torch.sigmoid(self.lin(h, p + "b"))
        g = torch.exp(-self.w(p + "A_log").exp() * torch.nn.functional.softplus(self.lin(h, p + "a") + self.w(p + "dt_bias")))
        S, o = h.new_zeros((H, D, V)), h.new_empty((T, H, V))
        for t in range(T):
            S = g[t][:, None, None] * S
            u = beta[t][:, None] * (v[t] - torch.matmul(k[t][:, None], S)[:, 0])
            S = S + k[t][:, :, None] * u[:, None, :]
            o[t] = torch.matmul(q[t][:, None], S)[:, 0]
        o = self.rms(o, p + "norm").reshape(T, -1) * silu(self.lin(h, p + "g"))
        return self.lin(o, p + "o")

    def retention(self, h, p, m):
        T, H, D, V = len(h), m["heads"], m["dim"], m["vdim"]
        q, k = (_rotate(self.lin(h, p + n).view(T, H, D), m["rot"]["base"], m["rot"]["dims"], True) for n in "qk")
        decay = torch.tensor(m["decay"], dtype=h.dtype, device=h.device).log().expand(T, H)
        o = _rms(_decayed_sum(q, k * D ** -0.5, self.lin(h, p + "v").view(T, H, V), decay), self.eps)
        return self.lin(o.reshape(T, -1) * torch.nn.functional.silu(self.lin(h, p + "g")), p + "o")

    def lightning(self, h, p, m, i):
        T, H, D, V = len(h), m["heads"], m["dim"], m["vdim"]
        q, k, v = (torch.nn.functional.silu(self.lin(h, p + n)).view(T, H, -1) for n in "qkv")
        decay = torch.tensor(m["decay"], dtype=h.dtype, device=h.device).log().expand(T, H)
        o = self.rms(_decayed_sum(q, k, v, decay).reshape(T, -1), p + "norm")
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def channel_delta(self, h, p, m):
        T, H, D = len(h), m["heads"], m["dim"]
        r, k, v = (self.lin(h, p + n).view(T, H, D) for n in "rkv")
        low = self.lin(torch.tanh(self.lin(h, p + "w1")), p + "w2") + self.w(p + "w0")
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(low)).view(T, H, D, 1)
        u = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        away = torch.sigmoid(self.lin(h, p + "a") + self.w(p + "a.b")).view(T, H, D) * u
        S, o = h.new_zeros((H, D, D)), h.new_empty((T, H, D))
        for t in range(T):
            S = decay[t] * S - away[t][:, :, None] * torch.matmul(u[t][:, None], S) + k[t][:, :, None] * v[t][:, None, :]
            o[t] = torch.matmul(r[t][:, None], S)[:, 0]
        o = _rms(o, self.eps).reshape(T, -1) * self.w(p + "norm")
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def parallel(self, h, p, m, i):
        right = self.channel_delta if self.kind == "Dimelix" else self.retention
        return m["left_scale"] * self.attention(h, p + "left.", m["left"], i) + m["right_scale"] * right(h, p + "right.", m["right"])

    # ---- feed-forwards: rows of any sequences
    def dense(self, h, p, f):
        if self.kind == "Dimelix":
            z, a = self.lin(h, p + "up"), torch.nn.functional.softplus(self.w(p + "act"))
            neg = z.clamp(max=0.0)
            return self.lin(torch.where(z > 0, a[0] * z * z + 0.5 * z, (0.5 + a[1]) * (torch.expm1(neg) - neg) + 0.5 * z), p + "down")
        g, u = self.lin(h, p + "gate"), self.lin(h, p + "up")
        if self.kind == "Kufolorn" and "limit" not in f:
            return self.lin(torch.nn.functional.gelu(g, approximate="tanh") * u, p + "down")
        g, u = g.clamp(max=f["limit"]), u.clamp(-f["limit"], f["limit"])
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")

    def feed_forward(self, h, p, f):
        if f["kind"] == "dense":
            return self.dense(h, p, f)
        z = h @ self.w(p + "router").t()
        if self.kind == "Sogenex":
            two = lambda x, q: self.lin(torch.relu(self.lin(x, q + "up")) ** 2, q + "down")  # noqa: E731
            z = z + self.w(p + "router.b")
            y = _routed(h, f, lambda idx: torch.softmax(z.gather(1, idx), 1), z, lambda e, x: two(x, f"{p}e{e}."))
            return y + torch.sigmoid(self.lin(h, p + "shared.sg")) * two(h, p + "shared.")
        if self.kind == "Kufolorn":
            s = torch.softmax(z, 1)
            return _routed(h, f, lambda idx: s.gather(1, idx), s + self.w(p + "correction"), lambda e, x: self.dense(x, f"{p}e{e}.", f["expert"]))
        two = lambda x, q: self.lin(torch.nn.functional.gelu(self.lin(x, q + "up")), q + "down")  # noqa: E731
        s = torch.sigmoid(z)
        y = _routed(h, f, lambda idx: s.gather(1, idx), s, lambda e, x: two(x, f"{p}e{e}."), on_input=True)
        return y + two(h, p + "shared.") if f.get("shared") else y

    # ---- the model
    def qwen2_layer(self, xs, i):
        c, p = self.cfg, f"model.layers.{i}."
        H, G, D = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        for n, x in enumerate(xs):
            h = self.rms(x, p + "input_layernorm.weight")
            q, k, v = (self.lin(h, f"{p}self_attn.{a}_proj.weight") + self.w(f"{p}self_attn.{a}_proj.bias") for a in "qkv")
            q, k = (_rotate(a.view(len(x), -1, D), c["rope_theta"], D, True) for a in (q, k))
            x = x + self.lin(_attend(q, k, v.view(-1, G, D), D ** -0.5).reshape(len(x), H * D), p + "self_attn.o_proj.weight")
            for part in x.split(2048):
                h = self.rms(part, p + "post_attention_layernorm.weight")
                part += self.lin(torch.nn.functional.silu(self.lin(h, p + "mlp.gate_proj.weight")) * self.lin(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
            xs[n] = x
        return xs

    def layer(self, x, i):
        L, p = self.cfg["layers"][i], f"l{i}."
        mix, m, f = getattr(self, L["type"]), L["mixer"], L["mlp"]
        if self.kind == "Kufolorn":
            x = x + self.norm(mix(x, p + "mix.", m, i), p + "norm1")
            return x + self.norm(self.feed_forward(x, p + "mlp.", f), p + "norm2")
        if self.kind == "Dimelix":                              # x [T, streams, W]
            for hc, nm, sub in (("hc1.", "norm1", lambda u: mix(u, p + "mix.", m, i)), ("hc2.", "norm2", lambda u: self.feed_forward(u, p + "mlp.", f))):
                u = self.norm(torch.einsum("s,tsw->tw", self.w(p + hc + "in"), x), p + nm)
                x = torch.einsum("sr,tsw->trw", self.w(p + hc + "mix"), x) + self.w(p + hc + "out")[None, :, None] * sub(u)[:, None, :]
            return x
        a = self.cfg.get("residual_mult", 1.0)
        x = x + a * mix(self.norm(x, p + "norm1"), p + "mix.", m, i)
        return x + a * self.feed_forward(self.norm(x, p + "norm2"), p + "mlp.", f)

    def logits(self, ids, wanted):
        """Per sequence the logits [wanted, vocab] at the wanted places."""
        c, table = self.cfg, "embed" if self.kind != "Qwen2" else "model.embed_tokens.weight"
        xs = [self.w(table)[torch.tensor(s, device=self.device)] for s in ids]
        out = []
        if self.kind == "Qwen2":
            tied = c["tie_word_embeddings"]
            if not tied:
                self.held.clear()
            for i in range(c["num_hidden_layers"]):
                keep = {table: self.held[table]} if tied else {}
                xs = self.qwen2_layer(xs, i)
                self.held = keep                                # a layer's matrices at a time
            for x, places in zip(xs, wanted):
                out.append(self.lin(self.rms(x[places], "model.norm.weight"), table if tied else "lm_head.weight"))
            return out
        for x, places in zip(xs, wanted):
            self.shared = {}
            x = x * (c.get("embedding") or {}).get("scale", 1.0)
            if self.kind == "Sogenex":
                i = torch.arange(0, x.shape[1], 2, dtype=x.dtype, device=x.device)
                a = torch.arange(len(x), dtype=x.dtype, device=x.device)[:, None] * 10000.0 ** (-i / x.shape[1])
                x = x + torch.stack([a.sin(), a.cos()], 2).reshape(len(x), -1)
            if self.kind == "Dimelix":
                x = x[:, None, :].expand(-1, c["streams"], -1)
            for i in _layer_order(c):
                x = self.layer(x, i)
            x = x.sum(1) if self.kind == "Dimelix" else x
            y = self.lin(self.norm(x[places], "final.norm"), "head" if "head" in self.known else "embed") * c.get("logit_scale", 1.0)
            cap = c.get("logit_softcap") or 0.0
            out.append(cap * torch.tanh(y / cap) if cap else y)
        return out


def exact(case, seed):
    if case["kind"] == "sample":
        return None                                             # whole numbers: the tokens
    cfg = config(case)
    ids = token_ids(case, seed, cfg)
    tokens = sum(len(s) for s in ids)
    known = tensors(cfg)
    layers = sum(_layer_work(cfg, i, known, 2)[1] for i in _layer_order(cfg))
    if layers * tokens > EXACT_FLOPS:
        return None
    steps = case.get("steps", 0)
    wanted = [list(range(len(s) - 1 - steps, len(s))) for s in ids]
    got = _Plain(cfg, seed, DTYPES[case["dtype"]][1], "cuda:0").logits(ids, wanted)
    rows = [torch.cat([g[j:j + 1] for g in got]) for j in range(steps + 1)]
    return rows if case["kind"] in ("answer", "prompt") else rows[0]
