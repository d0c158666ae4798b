"""What is timed when this library is made faster: steps of the Qwen2 decoder through `Model` and `Engine`.

The cases follow what a user's program does with them.  A serving program loads a model once, keeps an engine, and then
gives it prompts (one step for a batch of whole prompts, of which it wants the last place's logits) and decoding steps
(one token for each live sequence); a check or a trace replay runs a short request from its prompt to its last token.
The shapes are those of the catalog: the 7B, 1.5B and 32B ones in bfloat16 with the workloads that bench.py runs at them
(the 32B one with 8 of its 64 layers, so that three batches and the weights' two copies fit beside each other), the two
tiny ones with the workloads that the tests run at them, and the true 32-bit path at the 7B layers' sizes.  The catalog has the
other architectures as tiny shapes only, and a routed model's bfloat16 output is not comparable between two correct
implementations (a choice of experts that turns on a rounding changes a whole row), so they are not among the cases.
Drawing the next token is left to the caller for the same reason, and the decoding cases feed given tokens, as a replay does.

Weights are N(0, 0.02), norms 1 + N(0, 0.02), tokens uniform in the vocabulary; as in a trained model, and unlike a plain
random one, what a layer adds is small beside the stream it adds to (embeddings N(0, 1), the two products that add to the
stream divided by the square root of twice the depth), so that a rounding in one layer is not magnified by the next ones
(28 layers of N(0, 0.02) alone leave bfloat16 logits 6 to 8 percent off).  The weights of a shape are the same for every
seed, as a served model's are; the tokens come from the seed.  Lengths belong to the case.
"""
import gc
import json
import os
import random

import torch

import tq_kv_amd
from tq_kv_amd import Engine, Model

SHAPES = os.path.join(os.path.dirname(tq_kv_amd.__file__), "config", "shapes")
BF16, F32 = "bfloat16", "float32"
ROOM = 1024             # decoding steps a batch can go on for before it starts over from its prompts
MOST_STEP = 8192        # tokens one prompt step takes at most while a batch is brought up (the generation loop's own bound)


# -- the cases ---------------------------------------------------------------------------------------
def _case(name, kind, model, layers, dtype, lens, batch, steps=0, tune=False):
    """lens: "n" (every prompt has n tokens), "a,b,c" (one for each) or "a..b" (uniform, fixed by the case's batch)."""
    return {"name": name, "kind": kind, "model": model, "layers": layers, "dtype": dtype, "lens": lens, "batch": batch, "steps": steps, "tune": tune}


def listed():
    return [
        # The tests' first small configuration, as tests and a first try of the library run it: a ragged batch of three
        # prompts and eight decoding steps in 32 bits.  Nothing but launches and host work.
        _case("tiny a request", "request", "tiny-a", 2, F32, "5,11,17", 3, steps=8),
        # The second one: a sliding window, a group of three heads, four prompts of 1 to 33 tokens, ten steps.
        _case("tiny b request", "request", "tiny-b", 3, BF16, "1,7,20,33", 4, steps=10),
        # One user's chat at the 7B shape: a token at a time after 2048 tokens.
        _case("7b decode 1", "decode", "qwen2.5-7b", 28, BF16, "2048", 1),
        # The headline: eight sequences after prompts of 2048 tokens.
        _case("7b decode 8", "decode", "qwen2.5-7b", 28, BF16, "2048", 8),
        # A busy server: 64 sequences, each at a length of its own.
        _case("7b decode 64 ragged", "decode", "qwen2.5-7b", 28, BF16, "16..1024", 64),
        # The time to the first token of a few short chat prompts that came together.
        _case("7b short prompts", "prompt", "qwen2.5-7b", 28, BF16, "37,5,190", 3),
        # The headline's prompt pass, with the library's products tuned for its size as bench.py does it.
        _case("7b prompt 2048", "prompt", "qwen2.5-7b", 28, BF16, "2048", 1, tune=True),
        # A long document.
        _case("7b prompt 8000", "prompt", "qwen2.5-7b", 28, BF16, "8000", 1),
        # The 1.5B workload of bench.py: 32 prompts of unequal lengths in one step, then decoding.
        _case("1.5b prompts 32 ragged", "prompt", "qwen2.5-1.5b", 28, BF16, "16..1024", 32),
        _case("1.5b decode 32 ragged", "decode", "qwen2.5-1.5b", 28, BF16, "16..1024", 32),
        # The 32B workload of bench.py: 16 sequences after prompts of 512 tokens.
        _case("32b decode 16", "decode", "qwen2.5-32b", 8, BF16, "512", 16),
        # The true 32-bit path at the 7B layers' sizes, as a check of the bfloat16 one runs it: a prompt and four steps.
        _case("7b float32 request", "request", "qwen2.5-7b", 4, F32, "300", 1, steps=4),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "tiny", "float32"])
    if kind == "tiny":
        model, layers, most = rng.choice([("tiny-a", 2, 100), ("tiny-b", 3, 80)])
        n, steps = rng.randint(1, 6), rng.randint(4, 12)
        return _drawn("request", model, layers, rng.choice([BF16, F32]), [rng.randint(1, most // 2) for _ in range(n)], steps)
    if kind == "float32":
        return _drawn("request", "qwen2.5-7b", 4, F32, [_log_int(rng, 3, 100) for _ in range(rng.randint(1, 3))], rng.randint(1, 4))
    model, layers = rng.choice([("qwen2.5-7b", 28), ("qwen2.5-7b", 28), ("qwen2.5-1.5b", 28), ("qwen2.5-32b", 8)])
    if kind == "decode":
        batch = _log_int(rng, 1, 100)
        longest = _log_int(rng, 24, max(24, min(2048, 40000 // batch)))
        return _drawn("decode", model, layers, BF16, [rng.randint(max(1, longest // 8), longest) for _ in range(batch)], 0)
    tokens = _log_int(rng, 8, 8000)
    n = rng.randint(1, max(1, min(16, tokens // 8)))
    cuts = sorted(rng.sample(range(1, tokens), n - 1))
    return _drawn("prompt", model, layers, BF16, [b - a for a, b in zip([0] + cuts, cuts + [tokens])], 0)


def _drawn(kind, model, layers, dtype, lens, steps):
    c = _case("", kind, model, layers, dtype, ",".join(map(str, lens)), len(lens), steps)
    del c["name"]
    return c


def _lens(case):
    if ".." in case["lens"]:
        lo, hi = map(int, case["lens"].split(".."))
        r = random.Random(case["batch"])
        return [r.randint(lo, hi) for _ in range(case["batch"])]
    lens = [int(n) for n in case["lens"].split(",")]
    return lens * case["batch"] if len(lens) == 1 else lens


def _config(case):
    with open(os.path.join(SHAPES, case["model"] + ".json")) as f:
        cfg = json.load(f)
    cfg["num_hidden_layers"] = case["layers"]
    cfg["max_position_embeddings"] = max(cfg["max_position_embeddings"], max(_lens(case)) + 64)
    return cfg


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == BF16 else torch.float32


# -- what a program keeps: one model, one engine ------------------------------------------------------
def _weights(cfg, dtype):
    """(name, tensor) of the whole model, made on the GPU; the same ones every time."""
    h, inter, d = cfg["hidden_size"], cfg["intermediate_size"], cfg["head_dim"]
    q, kv = cfg["num_attention_heads"] * d, cfg["num_key_value_heads"] * d
    g = torch.Generator(device="cuda").manual_seed(1)

    def made(*shape, std=0.02):
        return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=g)

    adds = 0.02 / (2 * cfg["num_hidden_layers"]) ** 0.5
    yield "model.embed_tokens.weight", made(cfg["vocab_size"], h, std=1.0)
    for i in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % i
        yield p + "input_layernorm.weight", made(h) + 1
        for name, n in (("q_proj", q), ("k_proj", kv), ("v_proj", kv)):
            yield p + "self_attn.%s.weight" % name, made(n, h)
            yield p + "self_attn.%s.bias" % name, made(n)
        yield p + "self_attn.o_proj.weight", made(h, q, std=adds)
        yield p + "post_attention_layernorm.weight", made(h) + 1
        yield p + "mlp.gate_proj.weight", made(inter, h)
        yield p + "mlp.up_proj.weight", made(inter, h)
        yield p + "mlp.down_proj.weight", made(h, inter, std=adds)
    yield "model.norm.weight", made(h) + 1
    if not cfg["tie_word_embeddings"]:
        yield "lm_head.weight", made(cfg["vocab_size"], h)


_serving = {"key": None, "model": None, "engine": None, "room": 0, "tuned": set()}


def _pages(n):
    return (n + 63) // 64 * 64


def _engine(case):
    """The engine of the case's shape: the one at hand, where it is that and has room for four batches of the case."""
    s, cfg = _serving, _config(case)
    key = json.dumps([cfg, case["dtype"]], sort_keys=True)
    if s["key"] != key:
        s.update(key=None, model=None, engine=None, room=0, tuned=set())
        gc.collect()
        torch.cuda.empty_cache()
        s["model"] = Model.from_config_dict(cfg, case["dtype"], "cuda").load(dict(_weights(cfg, _dtype(case))))
        torch.cuda.empty_cache()
        s["key"] = key
    more = {"decode": ROOM, "request": case["steps"], "prompt": 0}[case["kind"]]
    room = 4 * sum(_pages(n + more) for n in _lens(case))
    if s["engine"] is None or s["room"] < room:
        s["engine"] = None
        s["engine"], s["room"] = Engine(s["model"], max_tokens=room, max_slots=1024), room
    tokens = sum(_lens(case))
    if case["tune"] and tokens not in s["tuned"]:
        s["model"].tune_library(tokens)
        s["tuned"].add(tokens)
    return s["engine"]


class Batch:
    """A batch of requests and, while it is being decoded, its slots of the engine."""

    def __init__(self, case, seed):
        self.kind, self.steps = case["kind"], case["steps"]
        self.engine, self.slots, self.at = _engine(case), [], 0
        lens, vocab = _lens(case), self.engine.vocab_size
        self.room = ROOM if self.kind == "decode" else self.steps
        g = torch.Generator().manual_seed(seed)
        self.prompts = [torch.randint(0, vocab, (n,), generator=g).tolist() for n in lens]
        self.fed = torch.randint(0, vocab, (self.room, len(lens)), generator=g, dtype=torch.int32)
        self.next = self.fed.cuda()                 # on the device, where a sampler leaves them
        self.last = [[n - 1] for n in lens]
        if self.kind == "decode":
            self.bring_up()

    def bring_up(self):
        """All prompts into the cache, whole ones together while they fit one step."""
        self.close()
        self.slots, self.at = [self.engine.open() for _ in self.prompts], 0
        items, n = [], 0
        for slot, p in zip(self.slots, self.prompts):
            if items and n + len(p) > MOST_STEP:
                self.engine.step(items)
                items, n = [], 0
            items.append((slot, p, []))
            n += len(p)
        self.engine.step(items)

    def decode(self):
        """One token for every sequence; the logits live in the engine's memory until its next step."""
        out = self.engine.step([(s, [0], [0]) for s in self.slots], borrow=True, device_tokens=self.next[self.at])
        self.at += 1
        return out

    def close(self):
        while self.slots:
            self.engine.close(self.slots.pop())

    def __del__(self):
        try:
            self.close()
        except Exception:       # the interpreter is going down
            pass


def prepare(case, seed):
    return Batch(case, seed)


def run(b):
    """decode: one step of the live batch.  prompt: the batch's prompts in one step, from open to close.  request: the
    prompts and then the given tokens one by one, the logits of all of it."""
    if b.kind == "decode":
        if b.at == b.room:
            b.bring_up()
        return b.decode()
    b.slots, b.at = [b.engine.open() for _ in b.prompts], 0
    out = [b.engine.step([(s, p, w) for s, p, w in zip(b.slots, b.prompts, b.last)])]
    for _ in range(b.steps):
        out.append(b.decode().clone())
    b.close()
    return torch.stack(out) if b.steps else out[0]


# -- what a pass cannot do without --------------------------------------------------------------------
def _step_work(cfg, size, starts, news, wanted):
    """Bytes and operations of one step: the weights once, the embedding's rows, the earlier keys and values in, the new
    ones and the logits out; in the last layer only the wanted rows go past keys and values."""
    h, inter, d, v, layers = cfg["hidden_size"], cfg["intermediate_size"], cfg["head_dim"], cfg["vocab_size"], cfg["num_hidden_layers"]
    q, kv = cfg["num_attention_heads"] * d, cfg["num_key_value_heads"] * d
    tokens = sum(news)
    kv_part, rest = 2 * h * kv, 2 * h * q + 3 * h * inter
    params = layers * (kv_part + rest + q + 2 * kv + 2 * h) + h * v + h
    byts = size * (params + tokens * h + 2 * kv * layers * (sum(starts) + tokens)) + 4 * wanted * v
    flops = 2 * (tokens * layers * kv_part + (tokens * (layers - 1) + wanted) * rest + wanted * h * v)
    for i, (s, n) in enumerate(zip(starts, news)):
        for layer in range(layers):
            w = cfg["sliding_window"] if cfg.get("use_sliding_window") and layer >= cfg["max_window_layers"] else s + n
            rows = range(s, s + n) if layer < layers - 1 else range(s + n - 1, s + n)
            seen = sum(min(w, p + 1) for p in rows) if w < s + n else (rows[0] + rows[-1] + 2) * len(rows) // 2
            flops += 4 * q * seen
    return byts, flops


def work(case):
    cfg, lens = _config(case), _lens(case)
    size, n = 2 if case["dtype"] == BF16 else 4, len(lens)
    if case["kind"] == "decode":
        b, f = _step_work(cfg, size, lens, [1] * n, n)
        return {"bytes": b, "flops": f}
    b, f = _step_work(cfg, size, [0] * n, lens, n)
    for i in range(case["steps"]):      # every decoding step reads the weights again: its tokens follow from the step before
        more = _step_work(cfg, size, [m + i for m in lens], [1] * n, n)
        b, f = b + more[0], f + more[1]
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Measured against exact(): 32 bits 1.5e-7 to 6e-7; bfloat16 0.0016 (the tiny shape), 0.0026 (1.5B), 0.007 to 0.008
    # (7B), 0.011 (the 32B layers), the largest single value about 6 times as much.  Four times the larger ones.
    if case["dtype"] == F32:
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.03, "max": 0.2}


# -- the same in 64 bits ------------------------------------------------------------------------------
def _attend(q, k, v, window):
    """q [nh, n, d], k and v [nkv, n, d] of one sequence -> [n, nh d], one kv head at a time."""
    nh, n, d = q.shape
    group = nh // k.shape[0]
    i = torch.arange(n, device=q.device)
    hidden = (i[None, :] > i[:, None]) | (i[None, :] <= i[:, None] - window)
    out = torch.empty(n, nh, d, dtype=q.dtype, device=q.device)
    for kvh in range(k.shape[0]):
        for first in range(kvh * group, (kvh + 1) * group):
            s = (q[first] @ k[kvh].t()) / d ** 0.5
            s.masked_fill_(hidden, float("-inf"))
            out[:, first] = torch.softmax(s, dim=-1) @ v[kvh]
    return out.reshape(n, nh * d)


def exact(case, seed):
    """Whole sequences with plain torch in 64 bits; the rotation's tables are the 32-bit ones that the architecture defines."""
    cfg, lens = _config(case), _lens(case)
    more = 1 if case["kind"] == "decode" else case["steps"]
    n_layers, eps, d = cfg["num_hidden_layers"], cfg["rms_norm_eps"], cfg["head_dim"]
    if work(dict(case, kind="prompt"))["flops"] > 5e14:      # more than about 20 seconds in 64 bits
        return None
    g = torch.Generator().manual_seed(seed)
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g).tolist() for n in lens]
    fed = torch.randint(0, cfg["vocab_size"], (ROOM if case["kind"] == "decode" else case["steps"], len(lens)), generator=g, dtype=torch.int32)
    seqs = [p + fed[:more, i].tolist() for i, p in enumerate(prompts)]
    ends = [0]
    for s in seqs:
        ends.append(ends[-1] + len(s))
    at = torch.tensor([p for s in seqs for p in range(len(s))], device="cuda")
    inv = 1.0 / torch.pow(torch.tensor(float(cfg["rope_theta"])), torch.arange(0, d, 2, dtype=torch.float32) / d)
    angle = (torch.arange(max(map(len, seqs)), dtype=torch.float32)[:, None] * inv[None, :]).cuda()
    cos, sin = angle.cos().double()[at][:, None, :], angle.sin().double()[at][:, None, :]

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()

    def turned(x):
        a, b = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1).transpose(0, 1)

    def rows(f, x, step=4096):
        return torch.cat([f(x[r:r + step]) for r in range(0, len(x), step)])

    stream = _weights(cfg, _dtype(case))
    _, embed = next(stream)
    x = embed[torch.tensor([t for s in seqs for t in s], device="cuda")].double()
    if not cfg["tie_word_embeddings"]:
        del embed
    for layer in range(n_layers):
        windowed = cfg.get("use_sliding_window") and layer >= cfg["max_window_layers"]
        w = {}
        for _ in range(12):
            name, t = next(stream)
            w[name.split(".", 3)[3]] = t
        y = norm(x, w["input_layernorm.weight"])
        q, k, v = (y @ w["self_attn.%s.weight" % p].double().t() + w["self_attn.%s.bias" % p].double() for p in ("q_proj", "k_proj", "v_proj"))
        q, k, v = turned(q.reshape(len(x), -1, d)), turned(k.reshape(len(x), -1, d)), v.reshape(len(x), -1, d).transpose(0, 1)
        y = torch.cat([_attend(q[:, a:b], k[:, a:b], v[:, a:b], cfg["sliding_window"] if windowed else b - a) for a, b in zip(ends, ends[1:])])
        x = x + y @ w["self_attn.o_proj.weight"].double().t()
        y = norm(x, w["post_attention_layernorm.weight"])
        gate, up, down = (w["mlp.%s_proj.weight" % p].double().t() for p in ("gate", "up", "down"))
        x = x + rows(lambda r: (torch.nn.functional.silu(r @ gate) * (r @ up)) @ down, y)
    x = norm(x, next(stream)[1])
    # the rows whose logits run() returns: of a decoding step the last one, else the prompt's last and every one after it
    steps = [more] if case["kind"] == "decode" else range(more + 1)
    pick = torch.tensor([[a + n - 1 + j for a, n in zip(ends, lens)] for j in steps], device="cuda")
    head = embed if cfg["tie_word_embeddings"] else next(stream)[1]
    out = torch.cat([x[pick] @ head[r:r + 32768].double().t() for r in range(0, cfg["vocab_size"], 32768)], -1)
    return out if case["kind"] == "request" and case["steps"] else out[0]
