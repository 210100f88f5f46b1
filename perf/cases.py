"""The work that a user of this engine has it do, as cases that can be timed and checked.

A case is one call of a serving program into `axon_amd.load(...)`'s engine, with random weights: a prompt (in one step or
in portions), a decoding step of live requests, or a step that mixes both.  The sizes are those that bench.py and the tests
use: the layers of Qwen2.5-7B and 14B, a dense decoder of width 2,048, the smoke run's tiny decoder, and the Pikesun,
Zugutar and Bafavik designs at width 2,048 (between them every kind of mixer and feed-forward: grouped-query, latent, masked
and differential attention, gated recurrence, state-space scan, delta rule, linear attention, dense and routed experts).

A process keeps one loaded model, as a serving program does; a state is the requests and tokens of one caller of it.
"""
import gc
import hashlib
import math
import weakref

import torch

import axon_amd
from axon_amd.engine import StepEntry

WEIGHT_SEED, STD, GAIN_STD = 0, 0.02, 0.1
MAX_LEN = 16384          # positions that a request may reach
ROOM = 4096              # a conversation that has grown by this many positions starts over

# ---------------------------------------------------------------------------- the models


def _dense(layers, width, heads, kv_heads, dim, ff, vocab, theta, eps):
    return dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=layers, hidden_size=width,
                intermediate_size=ff, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=dim, vocab_size=vocab,
                max_position_embeddings=MAX_LEN, rope_theta=theta, rms_norm_eps=eps, tie_word_embeddings=False)


def _pikesun():
    rec = {"type": "rglru", "mixer": {"width": 2560, "blocks": 10, "conv": 4}}
    att = {"type": "latent_attention", "mixer": {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512,
                                                 "q_rank": 768, "rot": {"base": 10000.0, "dims": 64}, "scale": 192 ** -0.5,
                                                 "mask": {"size": 1024}}}
    moe = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": 704, "limit": 7.0},
           "shared": {"ff": 1408, "limit": 7.0}}
    layers = [dict(rec, mlp={"kind": "dense", "ff": 5632}), dict(att, mlp=moe), dict(rec, mlp=moe), dict(att, mlp=moe)]
    return {"architecture": "Pikesun", "embedding": {"scale": 1.0}, "layers": layers, "norm": {"eps": 1e-6},
            "residual_mult": 1.0, "vocab": 32000, "width": 2048}


def _zugutar():
    both = {"type": "parallel", "mixer": {
        "left": {"heads": 16, "kv_heads": 2, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 10000.0, "dims": 64}},
        "right": {"heads": 32, "vdim": 64, "state": 128, "groups": 2, "conv": 4, "norm_groups": 2}}}
    att = {"type": "attention", "mixer": {"heads": 16, "kv_heads": 2, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                                          "q_temp": {"coef": 0.1, "every": 1024}}}
    moe = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": 704}, "shared": {"ff": 1408}}
    return {"architecture": "Zugutar", "layers": [dict(both, mlp=moe), dict(att, mlp=moe), dict(both, mlp=moe)],
            "loop": {"start": 2, "stop": 3, "times": 2}, "logit_scale": 0.25, "norm": {"eps": 1e-6}, "vocab": 32000,
            "width": 2048}


def _bafavik():
    def att(heads, kv_heads, dim, vdim, **more):
        return {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "scale": dim ** -0.5, **more}
    rot, mlp = {"base": 10000.0, "dims": 64}, {"kind": "dense", "ff": 8448}
    pair_2 = {"type": "parallel_2", "mixer": {
        "left": att(8, 2, 128, 256, conv=4, rot=rot),
        "right": {"heads": 16, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}}}
    pair = {"type": "parallel", "mixer": {
        "left": att(16, 2, 128, 128, rot=rot),
        "right": {"heads": 16, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** -(4 + 6 * i / 16) for i in range(16)]},
        "left_scale": 0.7, "right_scale": 0.7}}
    diff = {"type": "attention", "mixer": att(8, 1, 64, 128, diff=0.3, mask={"size": 1536})}
    return {"architecture": "Bafavik", "embedding": {"scale": 1.0, "bigram": {"buckets": 32003, "mul_prev": 8191, "mul_cur": 131}},
            "layers": [dict(pair_2, mlp=mlp), dict(pair, mlp=mlp), dict(diff, mlp=mlp)],
            "loop": {"start": 0, "stop": 1, "times": 2}, "residual_mult": 0.5, "logit_scale": 1.0, "norm": {"eps": 1e-6},
            "vocab": 32000, "width": 2048}


#: name -> (configuration, positions that the cache pool holds, live requests at most)
MODELS = {
    "qwen2.5-7b": (_dense(28, 3584, 28, 4, 128, 18944, 152064, 1000000.0, 1e-6), 320000, 200),
    "qwen2.5-14b, 8 layers": (_dense(8, 5120, 40, 8, 128, 13824, 152064, 1000000.0, 1e-5), 320000, 200),
    "dense 2048": (_dense(4, 2048, 16, 2, 128, 5632, 32000, 10000.0, 1e-6), 320000, 200),
    "tiny": (_dense(2, 64, 4, 2, 16, 176, 256, 10000.0, 1e-6), 4096, 8),
    "pikesun": (_pikesun(), 320000, 200),
    "zugutar": (_zugutar(), 320000, 200),
    "bafavik": (_bafavik(), 320000, 200),
}

# ---------------------------------------------------------------------------- the cases


def listed():
    return [
        # a three-token prompt to a test model, as `axon logits` is first tried: nothing but launches and host work
        dict(name="tiny 3 tokens", model="tiny", dtype="bfloat16", page=64, kind="prompt", requests=1, shortest=3, longest=3),
        # serving the headline model: eight conversations of unequal length, the usual load of one small server
        dict(name="7b decode 8 ragged", model="qwen2.5-7b", dtype="bfloat16", page=16, kind="decode", requests=8, shortest=301,
             longest=3907),
        # a full server: many conversations, mostly short
        dict(name="7b decode 64 short", model="qwen2.5-7b", dtype="bfloat16", page=64, kind="decode", requests=64, shortest=64,
             longest=900),
        # a prompt of the headline benchmark's length in one step
        dict(name="7b prompt 2048", model="qwen2.5-7b", dtype="bfloat16", page=16, kind="prompt", requests=1, shortest=2048,
             longest=2048),
        # a long document in portions of the scheduler's token budget
        dict(name="7b prompt 6000 portions", model="qwen2.5-7b", dtype="bfloat16", page=64, kind="prompt", requests=1,
             shortest=6000, longest=6000, portion=2048),
        # continuous batching: prompts of unequal length fed beside 32 decoding conversations
        dict(name="14b mixed", model="qwen2.5-14b, 8 layers", dtype="bfloat16", page=16, kind="mixed", requests=4, shortest=97,
             longest=803, rows=32, rows_shortest=150, rows_longest=1024),
        # the 32-bit path, which shows what bfloat16 hides: scoring a prompt, and decoding a few conversations
        dict(name="dense fp32 prompt 777", model="dense 2048", dtype="float32", page=64, kind="prompt", requests=1, shortest=777,
             longest=777),
        dict(name="dense fp32 decode 5", model="dense 2048", dtype="float32", page=64, kind="decode", requests=5, shortest=100,
             longest=1500),
        # the other designs, prompts and decoding: several ragged prompts in a step, a single long one, conversations
        dict(name="pikesun prompt 2048", model="pikesun", dtype="bfloat16", page=64, kind="prompt", requests=1, shortest=2048,
             longest=2048),
        dict(name="pikesun decode 8", model="pikesun", dtype="bfloat16", page=64, kind="decode", requests=8, shortest=200,
             longest=2500),
        dict(name="zugutar prompts 3 ragged", model="zugutar", dtype="bfloat16", page=64, kind="prompt", requests=3,
             shortest=311, longest=1203),
        dict(name="bafavik decode 16", model="bafavik", dtype="bfloat16", page=64, kind="decode", requests=16, shortest=90,
             longest=1700),
    ]


def draw(rng):
    """A case of the same ranges: every model, prompts of 1 to some thousand tokens, decoding of 1 to 64 requests with
    contexts up to 4,096 positions, both page sizes; the dense decoder in both data types."""
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    model = rng.choice(["qwen2.5-7b", "qwen2.5-7b", "qwen2.5-14b, 8 layers", "dense 2048", "dense 2048", "pikesun", "zugutar",
                        "bafavik", "tiny"])
    dtype = "float32" if model == "dense 2048" and rng.random() < 0.75 else "bfloat16"
    case = dict(model=model, dtype=dtype, page=rng.choice([16, 64]))
    if model == "tiny":
        n = spread(1, 64)
        return dict(case, kind="prompt", requests=1, shortest=n, longest=n)
    kind = rng.choice(["prompt", "prompt", "decode", "decode", "mixed"])
    most = 1024 if dtype == "float32" else 4096
    if kind == "prompt":
        requests = rng.choice([1, 1, 2, 3, 5])
        longest = max(1, spread(8, most) // requests)
        return dict(case, kind=kind, requests=requests, shortest=rng.randint(max(1, longest // 4), longest), longest=longest)
    if kind == "decode":
        requests = spread(1, 64)
        longest = spread(16, min(4096, 32768 // requests))
        return dict(case, kind=kind, requests=requests, shortest=max(1, int(longest * rng.uniform(0.1, 1.0))), longest=longest)
    requests, rows = rng.randint(1, 4), spread(1, 48)
    longest, rows_longest = max(1, spread(16, most // 2) // requests), spread(16, 1500)
    return dict(case, kind=kind, requests=requests, shortest=rng.randint(max(1, longest // 4), longest), longest=longest,
                rows=rows, rows_shortest=max(1, rows_longest // 5), rows_longest=rows_longest)


def _lengths(n, shortest, longest):
    """n lengths spread over their logarithm, the long and the short in turn."""
    if n == 1:
        return [longest]
    even = [int(round(shortest * (longest / shortest) ** (i / (n - 1)))) for i in range(n)]
    return [even[i // 2] if i % 2 else even[n - 1 - i // 2] for i in range(n)]


def _prompt_lengths(case):
    return _lengths(case["requests"], case["shortest"], case["longest"]) if case["kind"] != "decode" else []


def _row_lengths(case):
    """The context of every conversation that a decoding row belongs to."""
    if case["kind"] == "decode":
        return _lengths(case["requests"], case["shortest"], case["longest"])
    return _lengths(case["rows"], case["rows_shortest"], case["rows_longest"]) if case["kind"] == "mixed" else []


def _vocab(model):
    c = MODELS[model][0]
    return c.get("vocab_size") or c["vocab"]


STEPS = 64               # next tokens that a caller has for every conversation, taken round and round


def _tokens(case, seed):
    """(tokens of the new prompts, of the conversations so far, next tokens a step), from the seed alone."""
    g = torch.Generator().manual_seed(int(seed))
    vocab = _vocab(case["model"])

    def some(n):
        return torch.randint(0, vocab, (n,), generator=g).tolist()
    prompts, rows = [some(n) for n in _prompt_lengths(case)], [some(n) for n in _row_lengths(case)]
    return prompts, rows, [some(len(rows)) for _ in range(STEPS)] if rows else []


_loaded = {}             # the one model that this process keeps
_count = [0]


def _llm(case):
    key = (case["model"], case["dtype"], case["page"])
    if key not in _loaded:
        _loaded.clear()
        gc.collect()
        torch.cuda.empty_cache()
        config, positions, seqs = MODELS[case["model"]]
        _loaded[key] = axon_amd.load(config, dtype=case["dtype"], random_seed=WEIGHT_SEED, init_std=STD, page_size=case["page"],
                                     num_pages=positions // case["page"] + seqs, max_seqs=seqs, max_seq_len=MAX_LEN)
    return _loaded[key]


def _give_back(engine, ids):
    for rid in ids:
        engine.release(rid)


class State:
    """One caller: its engine, its live conversations and the tokens it will send."""

    def __init__(self, llm, case, seed):
        _count[0] += 1
        self.engine, self.portion = llm.engine, case.get("portion", 0)
        self.prompts, self.rows, self.steps = _tokens(case, seed)
        self.ids = [(_count[0], "row", i) for i in range(len(self.rows))]
        self.new_ids = [(_count[0], "new", i) for i in range(len(self.prompts))]
        self.end = weakref.finalize(self, _give_back, llm.engine, self.ids)
        self.at = 0
        self.begin()

    def begin(self):
        """The conversations so far, fed in steps of up to 4,096 tokens."""
        _give_back(self.engine, self.ids)
        entries, tokens = [], 0
        for rid, prompt in zip(self.ids, self.rows):
            if entries and tokens + len(prompt) > 4096:
                self.engine.step(entries)
                entries, tokens = [], 0
            entries.append(StepEntry(rid, prompt, []))
            tokens += len(prompt)
        if entries:
            self.engine.step(entries)
        self.at = 0


def prepare(case, seed):
    return State(_llm(case), case, seed)


def run(s):
    """The logits of the step's rows: every decoding row's, then the last place of every prompt."""
    if s.at == ROOM:
        s.begin()
    entries = []
    if s.ids:
        tokens = s.steps[s.at % STEPS]
        entries = [StepEntry(rid, [t], [0]) for rid, t in zip(s.ids, tokens)]
        s.at += 1
    if s.portion:
        for a in range(0, len(s.prompts[0]), s.portion):
            part = s.prompts[0][a:a + s.portion]
            last = a + s.portion >= len(s.prompts[0])
            out = s.engine.step([StepEntry(s.new_ids[0], part, [len(part) - 1] if last else [])], end=s.new_ids if last else [])
        return out
    entries += [StepEntry(rid, p, [len(p) - 1]) for rid, p in zip(s.new_ids, s.prompts)]
    return s.engine.step(entries, end=s.new_ids)


# ---------------------------------------------------------------------------- what a pass cannot do without


def _pairs(start, n, window):
    """Positions that n tokens from `start` on look at, all together."""
    return sum(min(p + 1, window) if window else p + 1 for p in (start, start + n - 1)) / 2 * n


def work(case):
    """Matrices that the step's tokens need once, the cache rows that they look at, states read and written, logits; two
    operations a weight and token, and a pair of positions' products in attention."""
    c = MODELS[case["model"]][0]
    e = 2 if case["dtype"] == "bfloat16" else 4
    spans = [(n, 1) for n in _row_lengths(case)] + [(0, n) for n in _prompt_lengths(case)]
    tokens, rows = sum(n for _, n in spans), len(spans)
    vocab = _vocab(case["model"])
    weights = flops = cache = state = 0

    def matrices(n):                        # n weights that every token meets
        nonlocal weights, flops
        weights += n
        flops += 2 * n * tokens

    def attention(per_pair, row, window=0):  # products a pair of positions, elements of a cached position
        nonlocal flops, cache
        flops += 2 * per_pair * sum(_pairs(s, n, window) for s, n in spans)
        cache += sum((min(s, window) if window else s) + n for s, n in spans) * row * e

    def scan(elems):                         # a state's elements: read and written a request, 3 products a token
        nonlocal flops, state
        flops += 6 * elems * tokens
        state += 8 * elems * rows

    def experts(width, mlp, mats):
        nonlocal weights, flops
        router, ff = mlp["router"], mlp["expert"]["ff"]
        one = mats * ff * width
        weights += one * router["experts"] * (1 - (1 - router["top"] / router["experts"]) ** tokens)
        flops += 2 * one * router["top"] * tokens
        matrices(router["experts"] * width + mats * mlp["shared"]["ff"] * width)

    if "layers" not in c:
        width, layers = c["hidden_size"], c["num_hidden_layers"]
        h, kv, d, ff = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["intermediate_size"]
        matrices(layers * ((2 * h + 2 * kv) * d * width + 3 * ff * width))
        attention(layers * 2 * h * d, layers * 2 * kv * d)
    else:
        width, loop = c["width"], c.get("loop")
        for i, layer in enumerate(c["layers"]):
            times = loop["times"] if loop and loop["start"] <= i < loop["stop"] else 1
            before = weights
            for _ in range(times):
                m, mlp, kind = layer["mixer"], layer["mlp"], layer["type"]
                if kind == "rglru":
                    w = m["width"]
                    matrices(3 * w * width + 2 * w * w // m["blocks"])
                    scan(w)
                elif kind == "latent_attention":
                    h, k = m["heads"], m["dim"] + m["rot_dim"]
                    matrices(m["q_rank"] * (width + h * k) + (m["kv_rank"] + m["rot_dim"]) * width
                             + h * (m["dim"] + m["vdim"]) * m["kv_rank"] + 2 * h * m["vdim"] * width)
                    attention(h * (k + m["vdim"]), m["kv_rank"] + m["rot_dim"], m["mask"]["size"])
                for side in ([m["left"]] if "left" in m else [m] if kind == "attention" else []):
                    h, g, d, dv = side["heads"], side["kv_heads"], side["dim"], side["vdim"]
                    maps = 2 if "diff" in side else 1
                    gate = h if _gates_heads(c, kind) else 0 if kind == "parallel" and "decay" in m["right"] else h * dv
                    matrices(((h + g) * d * maps + (g + h) * dv + gate) * width)
                    attention(h * maps * (d + dv), g * (d * maps + dv), side.get("mask", {}).get("size", 0))
                if "right" in m:
                    r = m["right"]
                    if "state" in r:
                        inner = r["heads"] * r["vdim"]
                        matrices((3 * inner + 2 * r["groups"] * r["state"] + r["heads"]) * width)
                        scan(inner * r["state"])
                    elif "decay" in r:
                        matrices(r["heads"] * (2 * r["dim"] + 3 * r["vdim"]) * width)
                        scan(r["heads"] * r["dim"] * r["vdim"])
                    else:
                        rank = max(16, width // 512 * 16)
                        key, val = r["heads"] * r["dim"], r["heads"] * r["vdim"]
                        matrices((2 * key + 2 * val + r["heads"] + 2 * rank) * width + rank * (key + val))
                        scan(key * r["vdim"])
                if mlp["kind"] == "dense":
                    matrices(2 * mlp["ff"] * width)
                else:
                    experts(width, mlp, 3)
            weights = before + (weights - before) / times      # a layer run again has its weights once
    head = vocab * width
    return {"bytes": (weights + head + tokens * width) * e + cache + state + rows * vocab * 4,
            "flops": flops + 2 * head * rows}


def _gates_heads(c, kind):
    return c["architecture"] == "Zugutar" and kind == "parallel"


def tolerance(case):
    """From the errors measured against the float64 values below: 4e-2 through the 28 layers of bfloat16 activations and
    2.7e-2 through the 8 wider ones (two orders of addition share most of it), 6e-3 through the smaller models, up to 2.4e-2
    where tokens choose experts, since a close call that goes the other way moves a whole row; 1.1e-6 in 32 bits."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    if case["model"] in ("pikesun", "zugutar"):
        return {"rel": 0.03, "max": 0.99}
    if case["model"].startswith("qwen2.5"):
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 0.02, "max": 0.2}


# ---------------------------------------------------------------------------- the same values in 64 bits
# Plain torch over the whole sequences laid one behind the other (`lens` are their lengths): no cache, nothing of the package.


class _Weights:
    """The tensors that `random_seed` stands for, drawn one at a time: N(0, 0.02), gains 1 + N(0, 0.1), rounded to the
    storage's type, as float64."""

    GAINS = ("norm", "norm1", "norm2", ".out", "ls1", "ls2", "layernorm.weight", "model.norm.weight")

    def __init__(self, dtype):
        self.storage = torch.bfloat16 if dtype == "bfloat16" else torch.float32

    def __call__(self, name, *shape):
        g = torch.Generator(device="cuda")
        g.manual_seed(int.from_bytes(hashlib.sha256(f"{WEIGHT_SEED}:{name}".encode()).digest()[:8], "little") & ((1 << 63) - 1))
        t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        t = t.mul_(GAIN_STD).add_(1.0) if name.endswith(self.GAINS) else t.mul_(STD)
        return t.to(self.storage).double()


def _unit(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _turned(x, lens, dims, base, neighbours=False):
    """x [N, heads, d]: the first `dims` places of every head turned by the token's position."""
    pos = torch.cat([torch.arange(n, device=x.device, dtype=torch.float64) for n in lens])
    angle = pos[:, None] * base ** (-torch.arange(0, dims, 2, device=x.device, dtype=torch.float64) / dims)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    first, rest = x[..., :dims], x[..., dims:]
    if neighbours:
        a, b = first[..., 0::2], first[..., 1::2]
        return torch.cat([torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2), rest], -1)
    a, b = first.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s, rest], -1)


def _attend(q, k, v, lens, scale, sees=None, sink=False):
    """q [N, H, d], k [N, G, d], v [N, G, dv]; `sees(i, j)` narrows what the causal mask leaves."""
    out, at, group = q.new_empty(q.shape[0], q.shape[1], v.shape[2]), 0, q.shape[1] // k.shape[1]
    for n in lens:
        i = torch.arange(n, device=q.device)
        ok = i[None, :] <= i[:, None]
        if sees is not None:
            ok &= sees(i[:, None], i[None, :])
        for h in range(q.shape[1]):
            s = (q[at:at + n, h] @ k[at:at + n, h // group].T * scale).masked_fill_(~ok, -math.inf)
            m = s.amax(-1, keepdim=True)
            m = m.clamp_min(0.0) if sink else m
            s = s.sub_(m).exp_()
            total = s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
            out[at:at + n, h] = s @ v[at:at + n, h // group] / total
        at += n
    return out


def _conv(x, taps, lens, bias=None):
    out, at, t = torch.empty_like(x), 0, taps.shape[1]
    for n in lens:
        p = torch.cat([x.new_zeros(t - 1, x.shape[1]), x[at:at + n]])
        out[at:at + n] = sum(p[j:j + n] * taps[:, j] for j in range(t))
        at += n
    return out if bias is None else out + bias


def _scan(lens, state, step, *rows):
    """`step(state, rows of one position of every sequence) -> (state, output)` over the sequences side by side."""
    def side_by_side(x):
        out, at = x.new_zeros(max(lens), len(lens), *x.shape[1:]), 0
        for b, n in enumerate(lens):
            out[:n, b] = x[at:at + n]
            at += n
        return out
    rows, outs = [side_by_side(r) for r in rows], []
    for t in range(max(lens)):
        state, o = step(state, *(r[t] for r in rows))
        outs.append(o)
    outs = torch.stack(outs)
    return torch.cat([outs[:n, b] for b, n in enumerate(lens)])


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _silu(x):
    return x * torch.sigmoid(x)


def _dense_stream(c, w, tokens, lens):
    width, ff, eps = c["hidden_size"], c["intermediate_size"], c["rms_norm_eps"]
    h, g, d = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
    theta = float(torch.tensor(c["rope_theta"], dtype=torch.float32))
    x = w("model.embed_tokens.weight", c["vocab_size"], width)[tokens]
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        y = _unit(x, eps) * w(p + "input_layernorm.weight", width)

        def proj(s, heads):
            name = f"{p}self_attn.{s}_proj."
            return (y @ w(name + "weight", heads * d, width).T + w(name + "bias", heads * d)).view(-1, heads, d)
        q, k, v = proj("q", h), proj("k", g), proj("v", g)
        o = _attend(_turned(q, lens, d, theta), _turned(k, lens, d, theta), v, lens, d ** -0.5)
        x = x + o.flatten(1) @ w(p + "self_attn.o_proj.weight", width, h * d).T
        y = _unit(x, eps) * w(p + "post_attention_layernorm.weight", width)
        y = _silu(y @ w(p + "mlp.gate_proj.weight", ff, width).T) * (y @ w(p + "mlp.up_proj.weight", ff, width).T)
        x = x + y @ w(p + "mlp.down_proj.weight", width, ff).T
    return _unit(x, eps) * w("model.norm.weight", width), w("lm_head.weight", c["vocab_size"], width)


def _experts(w, p, mlp, h, scored, unit):
    """`scored(z) -> (experts, their weights)`; `unit(gate, up)`; the weight is on the output, or on the input where scored
    says so."""
    width = h.shape[1]
    z = h @ w(p + "router", mlp["router"]["experts"], width).T
    chosen, share, on_input = scored(z, mlp["router"]["top"])

    def gated(name, ff, rows):
        mid = unit(rows @ w(name + "gate", ff, width).T, rows @ w(name + "up", ff, width).T)
        return mid @ w(name + "down", width, ff).T
    out = torch.zeros_like(h)
    for e in range(mlp["router"]["experts"]):
        t, at = (chosen == e).nonzero(as_tuple=True)
        if len(t):
            s = share[t, at][:, None]
            part = gated(f"{p}e{e}.", mlp["expert"]["ff"], h[t] * s if on_input else h[t])
            out[t] += part if on_input else part * s
    return out, gated(p + "shared.", mlp["shared"]["ff"], h)


def _pikesun_stream(c, w, tokens, lens):
    width, eps = c["width"], c["norm"]["eps"]
    x = w("embed", c["vocab"], width)[tokens] * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, m = f"l{i}.mix.", layer["mixer"]
        if layer["type"] == "rglru":
            n, blocks = m["width"], m["blocks"]
            y = _gelu(x @ w(p + "y", n, width).T + w(p + "y.b", n))
            u = _conv(x @ w(p + "x", n, width).T + w(p + "x.b", n), w(p + "conv", n, m["conv"]), lens, w(p + "conv.b", n))
            ub = u.view(-1, blocks, n // blocks).transpose(0, 1)

            def gate(s):
                z = ub @ w(p + s, blocks, n // blocks, n // blocks).transpose(1, 2).contiguous()
                return torch.sigmoid(z.transpose(0, 1) + w(p + s + ".b", blocks, n // blocks)).reshape(-1, n)
            a = torch.exp(-8.0 * gate("ra") * torch.nn.functional.softplus(w(p + "lam", n)))
            u = torch.sqrt(1.0 - a * a) * gate("ri") * u
            s = _scan(lens, u.new_zeros(len(lens), n), lambda s, a, u: (a * s + u,) * 2, a, u)
            mixed = (s * y) @ w(p + "o", width, n).T
        else:
            H, d, r, dv, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
            cq = _unit(x @ w(p + "dq", m["q_rank"], width).T, eps) * w(p + "dq.norm", m["q_rank"])
            q = (cq @ w(p + "uq", H * (d + r), m["q_rank"]).T).view(-1, H, d + r)
            down = x @ w(p + "dkv", rank + r, width).T
            latent = _unit(down[:, :rank], eps) * w(p + "dkv.norm", rank)
            turn = (lens, m["rot"]["dims"], m["rot"]["base"])
            q = torch.cat([q[..., :d], _turned(q[..., d:], *turn)], -1)
            key = _turned(down[:, None, rank:], *turn).expand(-1, H, -1)
            k = torch.cat([(latent @ w(p + "uk", H * d, rank).T).view(-1, H, d), key], -1)
            v = (latent @ w(p + "uv", H * dv, rank).T).view(-1, H, dv)
            size = m["mask"]["size"]
            o = _attend(q, k, v, lens, m["scale"], lambda i, j: i - j < size).flatten(1)
            mixed = (o * torch.sigmoid(x @ w(p + "g", H * dv, width).T)) @ w(p + "o", width, H * dv).T
        x = x + c["residual_mult"] * _unit(mixed, eps) * w(f"l{i}.norm1", width)
        p, mlp = f"l{i}.mlp.", layer["mlp"]
        if mlp["kind"] == "dense":
            y = _gelu(x @ w(p + "up", mlp["ff"], width).T) @ w(p + "down", width, mlp["ff"]).T
        else:
            limit = mlp["expert"]["limit"]

            def scored(z, top):
                best = z.topk(top, -1)
                return best.indices, best.values.softmax(-1), False

            def unit(g, u):
                g, u = g.clamp(max=limit), u.clamp(-limit, limit)
                return g * torch.sigmoid(1.702 * g) * (u + 1.0)
            y = sum(_experts(w, p, mlp, x, scored, unit))
        x = x + c["residual_mult"] * _unit(y, eps) * w(f"l{i}.norm2", width)
    return _unit(x, eps) * w("final.norm", width), w("head", c["vocab"], width)


def _heads(w, p, c, h, bias=False):
    """(q, k, v) [N, heads, d] of an attention's matrices."""
    def proj(s, n, d):
        y = h @ w(p + s, n * d, h.shape[1]).T
        return (y + w(p + s + ".b", n * d) if bias else y).view(-1, n, d)
    d = c["dim"] * (2 if "diff" in c else 1)
    return proj("q", c["heads"], d), proj("k", c["kv_heads"], d), proj("v", c["kv_heads"], c["vdim"])


def _zugutar_stream(c, w, tokens, lens):
    width, eps, loop = c["width"], c["norm"]["eps"], c["loop"]
    embed = w("embed", c["vocab"], width)
    x0 = x = embed[tokens]
    order = [(i, False) for i in range(loop["start"])]
    for k in range(loop["times"]):
        order += [(i, k > 0 and i == loop["start"]) for i in range(loop["start"], loop["stop"])]
    order += [(i, False) for i in range(loop["stop"], len(c["layers"]))]
    for i, again in order:
        x = x + x0 if again else x
        p, m = f"l{i}.mix.", c["layers"][i]["mixer"]
        h = _unit(x, eps) * (1.0 + w(f"l{i}.norm1", width))
        if c["layers"][i]["type"] == "attention":
            q, k, v = _heads(w, p, m, h)
            pos = torch.cat([torch.arange(n, device=x.device) for n in lens])
            steps = ((pos + 1) // m["q_temp"]["every"]).double()
            q = q * (1.0 + m["q_temp"]["coef"] * torch.log1p(steps))[:, None, None]
            o = _attend(q, k, v, lens, m["scale"]).flatten(1)
            y = (o * torch.sigmoid(h @ w(p + "g", o.shape[1], width).T)) @ w(p + "o", width, o.shape[1]).T
        else:
            a, r = m["left"], m["right"]
            q, k, v = _heads(w, p + "left.", a, h)
            turn = (lens, a["rot"]["dims"], a["rot"]["base"])
            q = _turned(_unit(q, eps) * w(p + "left.q.norm", a["dim"]), *turn)
            k = _turned(_unit(k, eps) * w(p + "left.k.norm", a["dim"]), *turn)
            o = _attend(q, k, v, lens, a["scale"], sink=True) * torch.sigmoid(h @ w(p + "left.g", a["heads"], width).T)[:, :, None]
            left = o.flatten(1) @ w(p + "left.o", width, a["heads"] * a["vdim"]).T
            p2, H, P, S, G = p + "right.", r["heads"], r["vdim"], r["state"], r["groups"]
            inner = H * P
            proj = h @ w(p2 + "in", 2 * inner + 2 * G * S + H, width).T
            z, xbc, dt = proj.split([inner, inner + 2 * G * S, H], -1)
            xbc = _silu(_conv(xbc, w(p2 + "conv", inner + 2 * G * S, r["conv"]), lens, w(p2 + "conv.b", inner + 2 * G * S)))
            u = xbc[:, :inner].reshape(-1, H, P)
            B = xbc[:, inner:inner + G * S].reshape(-1, G, S).repeat_interleave(H // G, 1)
            C = xbc[:, inner + G * S:].reshape(-1, G, S).repeat_interleave(H // G, 1)
            dt = torch.nn.functional.softplus(dt + w(p2 + "dt_bias", H), threshold=30.0)
            decay = torch.exp(-torch.exp(w(p2 + "A_log", H)) * dt)

            def step(s, a, u, B, C):
                s = a[..., None, None] * s + B[..., :, None] * u[..., None, :]
                return s, (C[..., None, :] @ s)[..., 0, :]
            y = _scan(lens, u.new_zeros(len(lens), H, S, P), step, decay, dt[..., None] * u, B, C)
            y = (y + w(p2 + "D", H)[:, None] * u).flatten(1) * _silu(z)
            y = _unit(y.view(-1, r["norm_groups"], inner // r["norm_groups"]), eps).flatten(1) * w(p2 + "norm", inner)
            right = y @ w(p2 + "o", width, inner).T
            y = 0.5 * (_unit(left, eps) * w(p + "left.out", width) + _unit(right, eps) * w(p + "right.out", width))
        p = f"l{i}.mlp."

        def scored(z, top):
            best = torch.sigmoid(z).topk(top, -1)
            return best.indices, best.values, True
        routed, shared = _experts(w, p, c["layers"][i]["mlp"], h, scored, lambda g, u: _silu(g) * u)
        x = x + y + routed + torch.sigmoid(h @ w(p + "shared.sg", 1, width).T) * shared
    return _unit(x, eps) * (1.0 + w("final.norm", width)), embed * c["logit_scale"]


def _bafavik_stream(c, w, tokens, lens):
    width, eps, loop, mult = c["width"], c["norm"]["eps"], c["loop"], c["residual_mult"]
    pairs = c["embedding"]["bigram"]
    first = torch.zeros_like(tokens, dtype=torch.bool)
    first[torch.tensor([sum(lens[:b]) for b in range(len(lens))], device=tokens.device)] = True
    bucket = (tokens.roll(1) * pairs["mul_prev"] + tokens * pairs["mul_cur"]) % pairs["buckets"]
    x = w("embed", c["vocab"], width)[tokens] * c["embedding"]["scale"]
    x = x + w("bigram", pairs["buckets"] + 1, width)[torch.where(first, pairs["buckets"], bucket)]
    order = list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"]
    for i in order + list(range(loop["stop"], len(c["layers"]))):
        p, layer = f"l{i}.mix.", c["layers"][i]
        m = layer["mixer"]
        h = _unit(x, eps) * (1.0 + w(f"l{i}.norm1", width))
        before = torch.where(first[:, None], 0.0, h.roll(1, 0))
        h = h + (before - h) * w(f"l{i}.shift", width)
        if layer["type"] == "attention":
            q, k, v = _heads(w, p, m, h, bias=True)
            d, size = m["dim"], m["mask"]["size"]
            a1, a2 = (_attend(q[..., s:s + d], k[..., s:s + d], v, lens, m["scale"], lambda i, j: i // size == j // size)
                      for s in (0, d))
            dot = [torch.exp((w(p + f"lq{n}", d) * w(p + f"lk{n}", d)).sum()) for n in (1, 2)]
            o = (_unit(a1 - (dot[0] - dot[1] + m["diff"]) * a2, eps) * (1.0 - m["diff"])).flatten(1)
            y = (o * torch.sigmoid(h @ w(p + "g", o.shape[1], width).T)) @ w(p + "o", width, o.shape[1]).T
        elif layer["type"] == "parallel":
            a, r = m["left"], m["right"]
            q, k, v = _heads(w, p + "left.", a, h, bias=True)
            turn = (lens, a["rot"]["dims"], a["rot"]["base"])
            o = _attend(_unit(_turned(q, *turn), eps), _unit(_turned(k, *turn), eps), v, lens, a["scale"]).flatten(1)
            left = o @ w(p + "left.o", width, o.shape[1]).T + w(p + "left.o.b", width)
            q, k, v = (_silu(t) for t in _heads(w, p + "right.", dict(r, kv_heads=r["heads"]), h))
            decay = torch.tensor(r["decay"], dtype=torch.float64, device=x.device)[:, None, None]

            def step(s, q, k, v):
                s = decay * s + k[..., :, None] * v[..., None, :]
                return s, (q[..., None, :] @ s)[..., 0, :]
            o = _scan(lens, q.new_zeros(len(lens), r["heads"], r["dim"], r["vdim"]), step, q, k, v).flatten(1)
            o = _unit(o, eps) * w(p + "right.norm", o.shape[1]) * torch.sigmoid(h @ w(p + "right.g", o.shape[1], width).T)
            y = m["left_scale"] * left + m["right_scale"] * (o @ w(p + "right.o", width, o.shape[1]).T)
        else:
            a, r = m["left"], m["right"]

            def convolved(q, c, s):
                n, d = q.shape[1:]
                return _conv(q.flatten(1), w(p + s + ".conv", n * d, c["conv"]), lens).view(-1, n, d)
            q, k, v = (convolved(t, a, "left." + s) for t, s in zip(_heads(w, p + "left.", a, h), "qkv"))
            turn = (lens, a["rot"]["dims"], a["rot"]["base"], True)
            o = _attend(_turned(q, *turn), _turned(k, *turn), v, lens, a["scale"]).flatten(1)
            left = (o * torch.sigmoid(h @ w(p + "left.g", o.shape[1], width).T)) @ w(p + "left.o", width, o.shape[1]).T
            p2, H, d, dv, rank = p + "right.", r["heads"], r["dim"], r["vdim"], max(16, width // 512 * 16)
            q, k, v = (_silu(convolved(t, r, "right." + s)) for t, s in zip(_heads(w, p2, r, h), "qkv"))
            q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
            k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            beta = torch.sigmoid(h @ w(p2 + "b", H, width).T)
            z = (h @ w(p2 + "a1", rank, width).T) @ w(p2 + "a2", H * d, rank).T + w(p2 + "dt_bias", H * d)
            z = torch.nn.functional.softplus(z, threshold=30.0).view(-1, H, d)
            g = torch.exp(-torch.exp(w(p2 + "A_log", H))[:, None] * z)

            def step(s, q, k, v, g, beta):
                s = g[..., None] * s
                u = beta[..., None] * (v - (k[..., None, :] @ s)[..., 0, :])
                s = s + k[..., :, None] * u[..., None, :]
                return s, (q[..., None, :] @ s)[..., 0, :]
            o = _scan(lens, q.new_zeros(len(lens), H, d, dv), step, q, k, v, g, beta)
            o = (_unit(o, eps) * w(p2 + "norm", dv)).flatten(1)
            o = o * torch.sigmoid((h @ w(p2 + "g1", rank, width).T) @ w(p2 + "g2", H * dv, rank).T)
            right = o @ w(p2 + "o", width, H * dv).T
            y = 0.5 * (_unit(left, eps) * w(p + "left.out", width) + _unit(right, eps) * w(p + "right.out", width))
        x = x + mult * w(f"l{i}.ls1", width) * y
        h, ff = _unit(x, eps) * (1.0 + w(f"l{i}.norm2", width)), layer["mlp"]["ff"]
        y = torch.relu(h @ w(f"l{i}.mlp.up", ff, width).T) ** 2 @ w(f"l{i}.mlp.down", width, ff).T
        x = x + mult * w(f"l{i}.ls2", width) * y
    return _unit(x, eps) * (1.0 + w("final.norm", width)), w("head", c["vocab"], width) * c["logit_scale"]


STREAMS = {"pikesun": _pikesun_stream, "zugutar": _zugutar_stream, "bafavik": _bafavik_stream}


def exact(case, seed):
    _loaded.clear()                     # room for the weights in 64 bits
    prompts, rows, steps = _tokens(case, seed)
    sequences = [r + [t] for r, t in zip(rows, steps[0] if steps else [])] + prompts
    lens = [len(s) for s in sequences]
    tokens = torch.tensor([t for s in sequences for t in s], device="cuda")
    last = torch.tensor(lens, device="cuda").cumsum(0) - 1
    stream = STREAMS.get(case["model"], _dense_stream)
    x, head = stream(MODELS[case["model"]][0], _Weights(case["dtype"]), tokens, lens)
    return x[last] @ head.T
