"""Steps of small models in one launch (csrc/small_step.hip) against the same steps through the kernels of larger ones: in float32 the same
bits, in bfloat16 as far apart as its roundings make two orders of summation.  Shapes with 16 to 64 values a head, widths that are and
are not whole steps of the matrix cores, more tiles than waves; steps of 1 to 64 rows on both sides of every change of the kernel."""
import pytest
import torch

import helpers
from tq_kv_amd import POLICY, Engine, Model

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def shape(hidden, inter, heads, kv_heads, head_dim, layers, vocab=97, window=None, tied=False):
    cfg = dict(helpers.TINY_A, hidden_size=hidden, intermediate_size=inter, num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim,
               num_hidden_layers=layers, vocab_size=vocab, tie_word_embeddings=tied, max_position_embeddings=256)
    if window:
        cfg.update(use_sliding_window=True, sliding_window=window, max_window_layers=1)
    return cfg


SHAPES = {
    "a": helpers.TINY_A, "b": helpers.TINY_B,
    "one head": shape(32, 32, 1, 1, 32, 1, vocab=16),
    "more tiles than waves": shape(96, 288, 4, 2, 64, 2, vocab=700, window=70),
    "wide": shape(160, 192, 5, 5, 32, 3, tied=True),
    "no whole step of k": shape(48, 80, 4, 2, 20, 2),              # float32 alone: bfloat16 takes 32 k at a time
    "many layers": shape(32, 64, 2, 1, 16, 16),
}


def close(a, b, dtype, what):
    if dtype == "float32":
        assert torch.equal(a, b), what
    else:                # (one rounding in a few hundred differs by a step of 2^-8; two such runs stay within a tenth of the logits' spread)
        assert (a - b).abs().max() <= 0.1 * b.std(), what


def steps(eng, vocab, count):
    """Prompts of several lengths, a chunk after them, single tokens from the host and from the device, wanted places out of order and none."""
    out, slots = [], [eng.open() for _ in range(3)]
    tok = lambda n, s: helpers.random_tokens(n, vocab, s)
    out.append(eng.step([(slots[0], tok(count, 1), [count - 1, 0] if count > 1 else [0])]))
    out.append(eng.step([(slots[1], tok(1, 2), [0]), (slots[0], tok(min(7, 65 - count), 3), [])]))
    out.append(eng.step([(slots[2], tok(9, 4), [8, 3]), (slots[1], tok(3, 5), [2])]))
    for i in range(3):
        dev = torch.tensor(tok(3, 10 + i), dtype=torch.int32, device=DEV) if i else None
        out.append(eng.step([(s, [t], [0]) for s, t in zip(slots, tok(3, 10 + i))], device_tokens=dev))
    borrowed = eng.step([(s, [1], [0]) for s in slots], borrow=True).clone()
    out.append(borrowed)
    for s in slots:
        eng.close(s)
    eng.cache.check()
    return out


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_the_step_in_one_launch_equals_the_kernels_of_larger_models(name, dtype):
    cfg = SHAPES[name]
    model = Model.random(cfg, seed=3, dtype=dtype, device=DEV)
    for count in [1, 2, 15, 16, 17, 31, 32, 33, 48, 61, 64]:
        got = steps(Engine(model, max_tokens=1024), cfg["vocab_size"], count)
        old = POLICY["small"]
        POLICY["small"] = False
        try:
            want = steps(Engine(model, max_tokens=1024), cfg["vocab_size"], count)
        finally:
            POLICY["small"] = old
        for i, (a, b) in enumerate(zip(got, want)):
            close(a, b, dtype, "%s, prompt of %d, step %d" % (name, count, i))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_several_pages_and_a_window_across_them(dtype):
    cfg = SHAPES["more tiles than waves"]
    model = Model.random(cfg, seed=4, dtype=dtype, device=DEV)
    tokens = helpers.random_tokens(210, cfg["vocab_size"], 9)

    def run():
        eng = Engine(model, max_tokens=512)
        s, out = eng.open(), []
        for a in range(0, 192, 48):
            out.append(eng.step([(s, tokens[a:a + 48], [47, 20, 0])]))
        for t in tokens[192:]:
            out.append(eng.step([(s, [t], [0])]))
        return torch.cat(out)

    got = run()
    POLICY["small"] = False
    try:
        want = run()
    finally:
        POLICY["small"] = True
    close(got, want, dtype, "several pages")
