"""Steps of small models in one launch (csrc/small_step.hip) against the same steps through the kernels of larger ones: the same bits.  Shapes with 16 to
64 values a head, widths that are and are not whole steps of the matrix cores, more tiles than waves, K that other kernels deal out to
waves or cut into pieces; steps of 1 to 64 rows on both sides of every change of the kernels that the step stands for.  Which way a step went is counted."""
import ctypes

import pytest
import torch

import helpers
import test_kernel_library
from tq_kv_amd import POLICY, Engine, Model, kernels, tracing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64


def shape(hidden, inter, heads, kv_heads, head_dim, layers, vocab=97, window=None, tied=False):
    cfg = dict(helpers.TINY_A, hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim,
               num_hidden_layers=layers, vocab_size=vocab, tie_word_embeddings=tied, max_position_embeddings=256)
    if window:
        cfg.update(use_sliding_window=True, sliding_window=window, max_window_layers=1)
    return cfg


# (and the most rows whose stream and products fit the unit's LDS, float32 and bfloat16)
SHAPES = {
    "a": (helpers.TINY_A, 64, 64), "b": (helpers.TINY_B, 64, 64),
    "one head": (shape(32, 32, 1, 1, 32, 1, vocab=16), 64, 64),
    "more tiles than waves": (shape(96, 224, 3, 1, 64, 2, vocab=700, window=70), 48, 48),
    "wide": (shape(160, 192, 5, 5, 32, 3, tied=True), 32, 32),
    "k dealt out to waves": (shape(256, 512, 4, 2, 64, 2, window=9), 19, 0),                # (bfloat16 keeps the order of the kernels that deal it out)
    "k in pieces": (shape(64, 1024, 2, 1, 32, 2), 16, 0),
    "many heads": (shape(32, 32, 28, 4, 8, 2, window=40), 48, 64),
    "more heads than a tile": (shape(32, 32, 20, 1, 32, 2, window=40), 16, 0),
    "no whole step of k": (shape(48, 80, 4, 2, 20, 2), 64, 0),              # float32 alone: bfloat16 takes 32 k at a time
    "many layers": (shape(32, 64, 2, 1, 16, 16), 64, 64),
}


class policy:
    def __init__(self, **values):
        self.values = values

    def __enter__(self):
        self.old = {n: POLICY[n] for n in self.values}
        POLICY.update(self.values)

    def __exit__(self, *_):
        POLICY.update(self.old)


class Steps:
    """An engine's steps, and how many of them the one launch should take."""

    def __init__(self, model, cfg, dtype, most, always):
        self.eng, self.most, self.expected = Engine(model, max_tokens=1024), most, 0
        self.always = always
        self.furthest = PAGE if dtype == "bfloat16" and cfg["head_dim"] in (32, 64) else 1 << 30       # those heads' attention is of one page there

    def __call__(self, items, **kw):
        self.expected += self.always and sum(len(t) for _, t, _ in items) <= self.most and max(self.eng.length(s) + len(t) for s, t, _ in items) <= self.furthest
        return self.eng.step(items, **kw)

    def done(self, slots):
        for s in slots:
            self.eng.close(s)
        self.eng.cache.check()
        assert self.eng.n_small_steps == self.expected


def steps(eng, vocab, count):
    """Prompts of several lengths, a chunk after them, single tokens from the host and from the device, wanted places out of order and none."""
    out, slots = [], [eng.eng.open() for _ in range(3)]
    tok = lambda n, s: helpers.random_tokens(n, vocab, s)
    out.append(eng([(slots[0], tok(count, 1), [count - 1, 0] if count > 1 else [0])]))
    out.append(eng([(slots[1], tok(1, 2), [0]), (slots[0], tok(min(7, 65 - count), 3), [])]))
    out.append(eng([(slots[2], tok(9, 4), [8, 3]), (slots[1], tok(3, 5), [2])]))
    for i in range(3):
        dev = torch.tensor(tok(3, 10 + i), dtype=torch.int32, device=DEV) if i else None
        out.append(eng([(s, [t], [0]) for s, t in zip(slots, tok(3, 10 + i))], device_tokens=dev))
    out.append(eng([(s, [1], [0]) for s in slots], borrow=True).clone())
    eng.done(slots)
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_the_step_in_one_launch_equals_the_kernels_of_larger_models(name, dtype):
    cfg, most = SHAPES[name][0], SHAPES[name][1 + (dtype == "bfloat16")]
    model = Model.random(cfg, seed=3, dtype=dtype, device=DEV)
    for count in [1, 2, 15, 16, 17, 31, 32, 33, 48, 58, 61, 64]:
        with policy(small_always=True):
            got = steps(Steps(model, cfg, dtype, most, True), cfg["vocab_size"], count)
        with policy(small=False):
            want = steps(Steps(model, cfg, dtype, most, False), cfg["vocab_size"], count)
        for i, (a, b) in enumerate(zip(got, want)):
            assert torch.equal(a, b), "%s, prompt of %d, step %d: %g of the values differ, by up to %g" % (
                name, count, i, (a != b).float().mean(), (a - b).abs().max())


@pytest.mark.parametrize("use_graphs", [True, False])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["a", "b", "one head", "more tiles than waves", "more heads than a tile", "many layers"])
def test_decoding_steps_of_many_sequences(name, dtype, use_graphs):
    """1 to 40 sequences of 1 to 60 positions (a page that is filled to its last place among them), some of their logits wanted."""
    cfg, most = SHAPES[name][0], SHAPES[name][1 + (dtype == "bfloat16")]
    model = Model.random(cfg, seed=5, dtype=dtype, device=DEV)

    def run(always):
        out = []
        for n in [1, 3, 15, 16, 17, 40]:
            s = Steps(model, cfg, dtype, most, always)
            s.eng = Engine(model, max_tokens=64 * 64, use_graphs=use_graphs)
            slots = [s.eng.open() for _ in range(n)]
            for i, slot in enumerate(slots):
                s([(slot, helpers.random_tokens(60 - 7 * i % 53, cfg["vocab_size"], i), [])])
            for k in range(4):
                out.append(s([(slot, [(5 * i + k) % cfg["vocab_size"]], [0] if (i + k) % 3 or n == 1 else []) for i, slot in enumerate(slots)]))
            s.done(slots)
        return out

    with policy(small_always=True):
        got = run(True)
    with policy(small=False):
        want = run(False)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), "%s, step %d: %g of the values differ, by up to %g" % (name, i, (a != b).float().mean(), (a - b).abs().max())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("head_dim", [64, 48, 32])
def test_several_pages_and_a_window_across_them(head_dim, dtype):
    cfg = shape(96, 96, 3, 1, head_dim, 2, vocab=700, window=70) if head_dim != 48 else shape(96, 96, 4, 2, head_dim, 2, vocab=700, window=70)
    chunk = 32 if head_dim == 64 else 48                    # (what fits the unit's LDS)
    model = Model.random(cfg, seed=4, dtype=dtype, device=DEV)
    tokens = helpers.random_tokens(210, cfg["vocab_size"], 9)

    def run(always):
        s = Steps(model, cfg, dtype, 64, always)
        s.eng = Engine(model, max_tokens=512)
        slot, out = s.eng.open(), []
        for a in range(0, 192, chunk):
            out.append(s([(slot, tokens[a:a + chunk], [chunk - 1, 20, 0])]))
        for t in tokens[192:]:
            out.append(s([(slot, [t], [0])]))
        s.done([slot])
        return torch.cat(out)

    with policy(small_always=True):
        got = run(True)
    with policy(small=False):
        want = run(False)
    assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_traced_step_gives_the_same_bits(dtype):
    """With ranges on the parts run one by one, so that they show: one launch less and nothing else."""
    model = Model.random(helpers.TINY_B, seed=3, dtype=dtype, device=DEV)
    names, got = [], []
    tracing.set_sink(lambda name: names.append(name.decode()), lambda: None)
    try:
        for on in (False, True):
            tracing.enable(on)
            eng = Engine(model, max_tokens=256)
            s = eng.open()
            got.append([eng.step([(s, helpers.random_tokens(12, helpers.TINY_B["vocab_size"], 1), [11, 0])]), eng.step([(s, [5], [0])])])
            assert eng.n_small_steps == (0 if on else 2) and ("attn" in names) == on
            eng.close(s)
    finally:
        tracing.enable(False)
        tracing.set_sink(None, None)
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_the_estimate_picks_the_faster_way():
    """Both sides of the rule's line, and a model that the kernel takes but that never pays."""
    model = Model.random(helpers.TINY_A, seed=3, dtype="bfloat16", device=DEV)
    for rows, small in ((1, 1), (64, 0)):
        eng = Engine(model, max_tokens=256)
        s = eng.open()
        eng.step([(s, [1] * rows, [0])])
        assert eng.n_small_steps == small
    wide = Model.random(shape(256, 512, 4, 2, 64, 4), seed=3, dtype="float32", device=DEV)
    eng = Engine(wide, max_tokens=256)
    eng.step([(eng.open(), [1], [0])])
    assert eng.n_small_steps == 0


# Weights through the ring in LDS: rows of an even and an odd number of 64 bytes, weights that end inside a unit of 1 KB, a ring that goes round inside a row and between layers, more and
# fewer than 128 k, features that fill no tile; a head that does not fit (and steps that want no logits, for which it does not count).
RING_SHAPES = {
    "a": helpers.TINY_A, "b": helpers.TINY_B,
    "long k": shape(144, 32, 2, 1, 16, 3, vocab=83),
    "odd": shape(48, 80, 3, 1, 16, 3, vocab=97),
    "small": shape(32, 32, 1, 1, 32, 5, vocab=33),
    "heads of 64": shape(64, 96, 2, 1, 64, 2, vocab=161),
    "no room for the head": shape(64, 160, 4, 2, 16, 2, vocab=600),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(RING_SHAPES))
def test_decoding_steps_with_their_weights_brought_into_lds(name, dtype):
    """1 to 13 sequences (4 and 12 are the most with a ring), some or none of their logits wanted."""
    cfg = RING_SHAPES[name]
    if dtype == "bfloat16" and cfg["hidden_size"] % 32:
        pytest.skip("bfloat16 takes 32 k at a time")
    model = Model.random(cfg, seed=7, dtype=dtype, device=DEV)

    def run(always):
        out = []
        for n in [1, 2, 3, 4, 5, 12, 13]:
            s = Steps(model, cfg, dtype, 64, always)
            slots = [s.eng.open() for _ in range(n)]
            for i, slot in enumerate(slots):
                s([(slot, helpers.random_tokens(1 + 5 * i % 40, cfg["vocab_size"], i), [])])
            for i in range(4):
                tokens = helpers.random_tokens(n, cfg["vocab_size"], 50 + i)
                out.append(s([(slot, [t], [0] if i == 3 or (i and j % 2 == 0) else []) for j, (slot, t) in enumerate(zip(slots, tokens))]))
            s.done(slots)
        return out

    with policy(small_always=True):
        got = run(True)
    with policy(small=False):
        want = run(False)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), "%s, step %d" % (name, i)


PAGE_SHAPES = {
    "heads of 4": shape(32, 32, 8, 8, 4, 2), "heads of 20": shape(48, 80, 4, 2, 20, 2, window=5), "heads of 16": shape(32, 32, 4, 2, 16, 2, window=33),
    "heads of 48": shape(96, 96, 2, 1, 48, 2), "heads of 64": shape(64, 64, 3, 1, 64, 2, window=17), "many heads on one": shape(32, 32, 20, 1, 16, 2),
}


def goes_by_units(cfg, lens, end):
    """Whether a float32 step of so many new tokens a sequence, up to `end` positions, has its attention by units of columns."""
    step = test_kernel_library.small_step(act_dtype=0, n_layers=cfg["num_hidden_layers"], hidden=cfg["hidden_size"], n_heads=cfg["num_attention_heads"], n_kv_heads=cfg["num_key_value_heads"],
                                          head_dim=cfg["head_dim"], inter=cfg["intermediate_size"], vocab=cfg["vocab_size"], n_rows=sum(lens), n_seqs=len(lens),
                                          decode=int(max(lens) == 1), max_end=end)
    for i in range(len(lens) + 1):
        step.ints[i] = sum(lens[:i])
    return bool(kernels.library().tqk_small_step_pages(ctypes.byref(step)))


@pytest.mark.parametrize("name", list(PAGE_SHAPES))
def test_float32_attention_within_a_page(name):
    """Several sequences of one step, up to the page's last place and one past it; columns that fill no tile and more than one; windows; both ways to have the attention."""
    cfg = PAGE_SHAPES[name]
    model = Model.random(cfg, seed=11, dtype="float32", device=DEV)
    ways = []

    def run(always):
        out = []
        for lens in [(1,), (1, 16, 17), (33, 2), (20, 20, 24), (63,), (64,)]:
            eng, n_steps = Engine(model, max_tokens=1024), 0
            slots = [eng.open() for _ in lens]
            tok = lambda n, seed: helpers.random_tokens(n, cfg["vocab_size"], seed)

            def step(items):
                nonlocal n_steps
                n_steps += 1
                ways.append(goes_by_units(cfg, [len(t) for _, t, _ in items], max(eng.length(s) + len(t) for s, t, _ in items)))
                out.append(eng.step(items))

            if sum(lens) <= 48 or cfg["num_attention_heads"] * cfg["head_dim"] < 192:             # (what fits the unit's LDS)
                step([(s, tok(n, n), list(range(n))) for s, n in zip(slots, lens)])
            else:
                for s, n in zip(slots, lens):
                    for a in range(0, n, 32):
                        step([(s, tok(n, n)[a:a + 32], [0])])
            for i in range(2):                                      # a chunk, then single tokens, one of them past the page
                step([(s, tok(1 + 4 * (i == 0 and n < 60), i), [0]) for s, n in zip(slots, lens)])
            assert eng.n_small_steps == (n_steps if always else 0)
        return out

    with policy(small_always=True):
        got = run(True)
    with policy(small=False):
        want = run(False)
    assert 8 <= sum(ways) // 2 <= len(ways) // 2 - 3, "%d of %d steps by units" % (sum(ways) // 2, len(ways) // 2)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), "%s, step %d: %g of the values differ, by up to %g" % (name, i, (a != b).float().mean(), (a - b).abs().max())


def same_numbers(a, b):
    return torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


@pytest.mark.parametrize("head_dim", [16, 20, 32, 48, 64])
@pytest.mark.parametrize("window", [None, 3])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), "one element"])
def test_float32_attention_within_a_page_keeps_what_is_not_finite_to_the_columns_that_see_it(value, window, head_dim):
    """One token's embedding is not finite, or one element of its value in the first layer: every position before it, and every one whose window is past it in all layers, has the bits
    that it has in the other kernels."""
    cfg = shape(32, 32, 4, 2, 16, 2, window=window) if head_dim == 16 else shape(64, 64, 4, 2, head_dim, 2, window=window)
    if window:
        cfg["max_window_layers"] = 0
    weights = model_weights(cfg)
    if value == "one element":
        # (the token alone has something in its first place, eight in its normed row; that times 1e38 is beyond float32, in one of an element's neighbours only)
        table = weights["model.embed_tokens.weight"]
        table[:, 0], table[5] = 0.0, 0.0
        table[5, 0] = 1.0
        v = weights["model.layers.0.self_attn.v_proj.weight"]
        v[head_dim + head_dim // 2 + 1, 0] = 1e38
    else:
        weights["model.embed_tokens.weight"][5] = value
    model = Model.from_config_dict(cfg, "float32", DEV).load(weights)
    tokens = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17]
    assert goes_by_units(cfg, [17, 4], 17)

    def run(small):
        eng = Engine(model, max_tokens=256)
        a, b = eng.open(), eng.open()
        out = eng.step([(a, tokens, list(range(17))), (b, tokens[:4], [3])])
        assert eng.n_small_steps == small
        return out

    with policy(small_always=True):
        got = run(1)
    with policy(small=False):
        want = run(0)
    assert torch.isfinite(want[:4]).all() and torch.isfinite(want[17]).all() and not torch.isfinite(want[4]).any()
    assert torch.isfinite(want[16]).all() == bool(window)
    assert same_numbers(got, want)


@pytest.mark.parametrize("where", ["weights", "weights and values", "products"])
@pytest.mark.parametrize("head_dim", [16, 20, 32, 64])
def test_subnormal_numbers_in_float32_steps(where, head_dim):
    """Values of 2^-130 and 2^-138 from subnormal weights, or of 2^-121 from ordinary ones, of which their products with the attention's weights are subnormal for some positions; the products behind
    bring them back.  Decoding steps of one to five sequences (with a ring up to four), chunks, attention by units and by queries: the bits of the other kernels, and not those without values."""
    cfg = shape(64, 96, 4, 2, head_dim, 2, vocab=97) if head_dim != 64 else shape(64, 96, 2, 1, 64, 2, vocab=97)

    def made(values):
        weights = model_weights(cfg)
        for i in range(2):
            p = "model.layers.%d." % i
            down = {"weights": 2.0 ** -128, "weights and values": 2.0 ** -136, "products": 2.0 ** -120}[where]
            weights[p + "self_attn.v_proj.weight"] *= down * values
            weights[p + "self_attn.v_proj.bias"] *= down * values
            weights[p + "self_attn.q_proj.weight"] *= 20.0                      # (weights of positions from 1 to 2^-20)
            weights[p + "self_attn.k_proj.weight"] *= 20.0
            weights[p + "self_attn.o_proj.weight"] *= 2.0 ** 125
            weights[p + "mlp.up_proj.weight"][:40] *= 2.0 ** -126               # (and the second half of an MLP)
            weights[p + "mlp.down_proj.weight"][:, :40] *= 2.0 ** 120
        return Model.from_config_dict(cfg, "float32", DEV).load(weights)

    def run(model):
        out, ways = [], []
        for n in (1, 2, 3, 4, 5):
            eng = Engine(model, max_tokens=1024)
            slots = [eng.open() for _ in range(n)]
            for lens in ([33 - 4 * i for i in range(n)] if n < 3 else [12] * n, [1] * n, [1] * n, [3] * n, [1] * n):
                ways.append(goes_by_units(cfg, lens, max(eng.length(s) + l for s, l in zip(slots, lens))))
                out.append(eng.step([(s, helpers.random_tokens(l, 97, len(out) + i), [l - 1]) for i, (s, l) in enumerate(zip(slots, lens))]))
            assert eng.n_small_steps == (5 if POLICY["small"] else 0)
        return torch.cat(out), ways

    model = made(1.0)
    with policy(small_always=True):
        got, ways = run(model)
    with policy(small=False):
        want, without = run(model)[0], run(made(0.0))[0]
    assert torch.isfinite(want).all() and len(set(ways)) == 2
    assert (want - without).abs().max() > 1e-4 * want.abs().max()
    assert torch.equal(got, want)


def model_weights(cfg, seed=13):
    """A whole model's tensors, N(0, 0.05), norms 1."""
    g = torch.Generator().manual_seed(seed)
    made = lambda *sizes: torch.randn(sizes, generator=g).mul_(0.05).to(DEV)
    h, q, kv, inter = cfg["hidden_size"], cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"], cfg["intermediate_size"]
    out = {"model.embed_tokens.weight": made(cfg["vocab_size"], h), "model.norm.weight": torch.ones(h, device=DEV), "lm_head.weight": made(cfg["vocab_size"], h)}
    for i in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % i
        out.update({p + "input_layernorm.weight": torch.ones(h, device=DEV), p + "post_attention_layernorm.weight": torch.ones(h, device=DEV),
                    p + "self_attn.o_proj.weight": made(h, q), p + "mlp.gate_proj.weight": made(inter, h), p + "mlp.up_proj.weight": made(inter, h), p + "mlp.down_proj.weight": made(h, inter)})
        for name, n in (("q", q), ("k", kv), ("v", kv)):
            out[p + "self_attn.%s_proj.weight" % name] = made(n, h)
            out[p + "self_attn.%s_proj.bias" % name] = made(n)
    return out
