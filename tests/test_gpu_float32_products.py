"""float32 products with large weights, whose numbers go through the matrix cores as three bfloat16 ones each (csrc/gemm_generic.hip): the
same bits whatever the number of rows (one kernel each for up to 4, 8 and 16 rows, four tiles for more), and no further from 64 bits than the float32
instructions are; infinities, NaN and numbers that overflow come out as float32 arithmetic gives them."""
import pytest
import torch

from tq_kv_amd import kernels as K

pytestmark = pytest.mark.gpu
ROWS = [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 130]


def operands(kind, m, n, k):
    """x and w of a kind: dense ones of several sizes, and rows that one value makes up, alone or by far."""
    g = torch.Generator(device="cuda").manual_seed(len(kind) + k)
    rand = lambda *s: torch.randn(s, device="cuda", generator=g)
    x, w = rand(m, k), rand(n, k)
    if kind == "one sign":
        x, w = x.abs(), w.abs()
    elif kind == "spread":
        x = x * 10 ** (torch.rand((m, k), device="cuda", generator=g) * 12 - 6)
    elif kind in ("one term", "one large term"):
        at = torch.arange(m, device="cuda")
        large = x[at, at * 7 % k]
        x = torch.zeros_like(x) if kind == "one term" else x * 1e-4
        x[at, at * 7 % k] = large if kind == "one term" else large * 1e4
    return x, w


@pytest.mark.parametrize("m", [8, 64])
@pytest.mark.parametrize("k", [1024, 3584, 18944])
@pytest.mark.parametrize("kind", ["normal", "one sign", "spread", "one term", "one large term"])
def test_no_further_from_64_bits_than_the_float32_instructions(kind, k, m):
    """The same rows and weights through the float32 instructions: slices of the weights that are too small to be taken apart.  Two ways to round the same sums differ by
    chance as well: of 64 rows by more than a thousand features a hundredth."""
    x, w = operands(kind, m, max(1024, (1 << 20) // k + 64), k)
    step = ((1 << 20) - 1) // k
    plain = torch.cat([product(x, w[a:a + step].contiguous(), None) for a in range(0, len(w), step)], 1)
    y, want = product(x, w, None), x.double() @ w.double().t()
    assert (y - want).norm() <= 1.01 * (plain - want).norm(), ((y - want).norm() / want.norm() * 2 ** 24, (plain - want).norm() / want.norm() * 2 ** 24)
    if kind == "one term":          # a product rounded once, and what the smaller parts' sum is cut off by, 2^-7 of that
        assert ((y - want).abs() / want.abs().clamp_min(1e-30)).max() <= (1 + 2 ** -5) * 2 ** -24


# (the exponents of x and w: sums below 2^-64 of numbers that bfloat16's range ends in, of subnormal ones, of products that are subnormal, and sums above the line)
@pytest.mark.parametrize("ex,ew", [(-100, 0), (-118, 0), (-118, 20), (-130, 0), (-70, -70), (-100, 34)])
@pytest.mark.parametrize("n,k", [(1024, 1024), (2049, 1540)])
def test_small_numbers(n, k, ex, ew):
    """No further from 64 bits than the float32 instructions, the same rows in every batch, and where all sums are below the line the float32 instructions' bits."""
    x, w = operands("normal", 130, n, k)
    x, w = x * 2.0 ** ex, w * 2.0 ** ew
    x[5], w[7] = 0.0, 0.0
    step = ((1 << 20) - 1) // k
    plain = torch.cat([product(x, w[a:a + step].contiguous(), None) for a in range(0, n, step)], 1)
    y, want = product(x, w, None), x.double() @ w.double().t()
    assert (y - want).norm() <= 1.01 * (plain - want).norm()
    if -140 < ex + ew < -80:        # (below, where float32 keeps a few bits of a sum, what they are by parts may be 0, which stands)
        assert torch.equal(y, plain)
    for m in ROWS:
        assert torch.equal(product(x[:m].contiguous(), w, None), y[:m]), m


def product(x, w, bias):
    y = torch.empty((x.shape[0], w.shape[0]), dtype=torch.float32, device="cuda")
    return K.gemm(x, w, bias, y)


# N, K: whole stages and chunks of k and not, one group of k and several, features that are no whole tiles, few blocks and many, just above the line
@pytest.mark.parametrize("n,k,bias", [(1024, 1024, True), (4608, 3584, True), (700, 18944, False), (5003, 1028, True), (2049, 516, False), (1030, 1088, False),
                                      (16390, 64, True), (262144, 4, False), (152064, 896, False)])
def test_rows_do_not_depend_on_the_batch_and_are_as_exact_as_float32_sums(n, k, bias):
    g = torch.Generator(device="cuda").manual_seed(n + k)
    assert n * k >= 1 << 20
    w = torch.randn((n, k), device="cuda", generator=g) * 0.02
    x = torch.randn((max(ROWS), k), device="cuda", generator=g) * torch.exp(torch.randn((max(ROWS), 1), device="cuda", generator=g))
    b = torch.randn((n,), device="cuda", generator=g) if bias else None
    whole = product(x, w, b)
    for m in ROWS:
        assert torch.equal(product(x[:m].contiguous(), w, b), whole[:m]), m
        assert torch.equal(product(x[-m:].contiguous(), w, b), whole[-m:]), m
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    # A float32 sum by chunks: within a chunk the sum of the largest products is cut off four times, 2^-23 of what is summed so far at most, and that of the others, a 128th of the
    # size, 28 times; they round once where they meet, and once for each of the chunks, groups and the bias, 2^-24, all independent: variances of 4 / 3 and 1 / 3 of 2^-48,
    # no more than sqrt(10) 2^-24 of the result's spread, and the same again for terms that cancel.
    spread = (x.double().norm(dim=1, keepdim=True) * w.double().norm(dim=1)) + (b.double().abs() if bias else 0)
    assert ((whole - want).abs() / spread).max() <= 8 * 2 ** -24
    assert (whole - want).norm() <= 2 * (10 ** 0.5) * 2 ** -24 * want.norm()


@pytest.mark.parametrize("n,k", [(2048, 1540), (1024, 3584)])
@pytest.mark.parametrize("m", [2, 7, 16, 40, 100])
def test_infinities_nan_and_overflow(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    x, w = torch.randn((m, k), device="cuda", generator=g), torch.randn((n, k), device="cuda", generator=g)
    x[0, 7], w[5, 9], w[6, k - 4] = float("inf"), float("-inf"), float("nan")
    # (64 bits do not overflow: these two numbers meet one row of x each, and nothing else that large)
    x[:, 3], w[:, 3], x[:, 11] = 0.0, 0.0, 0.0
    w[77, 3], x[m - 1, 3] = 3.3e38, 3.0e38                    # a product of its own beyond float32
    w[78, 11], x[m - 1, 11] = 3.39e38, 0.5                     # a number that a rounding to eight bits would make infinite
    y, want = product(x, w, None), (x.double() @ w.double().t()).float()
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(torch.isinf(y), torch.isinf(want))
    finite = torch.isfinite(want)
    assert torch.equal(torch.sign(y[~finite & ~torch.isnan(want)]), torch.sign(want[~finite & ~torch.isnan(want)]))
    torch.testing.assert_close(y[m - 1, 78], want[m - 1, 78])


@pytest.mark.parametrize("n,k", [(2048, 1540), (1024, 3584), (4608, 2048)])
def test_what_is_not_finite_changes_nothing_beside_it(n, k):
    """One row of x and one of w hold what is not finite (in the first group of k, in the last, in both), and everything else keeps the bits that
    it has without them, whatever the number of rows: the same tile's, the other groups' of the same sum, a row's alone."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.randn((130, k), device="cuda", generator=g), torch.randn((n, k), device="cuda", generator=g)
    clean = product(x, w, None)
    for bad_row, bad_feature, places in ((0, 5, [7]), (3, n - 1, [k - 2]), (9, 17, [1, k - 1])):
        xb, wb = x.clone(), w.clone()
        for p in places:
            xb[bad_row, p], wb[bad_feature, p] = float("inf"), float("nan")
        alone = product(xb[bad_row:bad_row + 1].contiguous(), wb, None)[0]
        for m in ROWS:
            y, rows = product(xb[:m].contiguous(), wb, None), torch.arange(m, device="cuda") != bad_row
            kept = torch.arange(n, device="cuda") != bad_feature
            assert torch.equal(y[rows][:, kept], clean[:m][rows][:, kept]), m
            assert not torch.isfinite(y[:, bad_feature]).any()
            if m > bad_row:
                assert torch.equal(y[bad_row].isnan(), alone.isnan()) and torch.equal(y[bad_row][~alone.isnan()], alone[~alone.isnan()]), m
    # a sum that overflows in float32 in one group of k and the other groups finite: the same for every number of rows
    x[1, :4], w[8, :4] = 2e19, 2e19
    one = product(x[1:2].contiguous(), w, None)[0]
    assert torch.isinf(one[8])
    for m in ROWS[1:]:
        assert torch.equal(product(x[:m].contiguous(), w, None)[1], one), m


# m, n, k, and how many blocks share K: a group each, two groups and a last one alone, two and none left, one block for all of K (400 to 767 tiles and more)
@pytest.mark.parametrize("m,n,k,shares", [(17, 3584, 18944, 19), (100, 3584, 18944, 10), (160, 4096, 11008, 6), (200, 7168, 5116, 3), (1000, 4608, 3584, 4),
                                          (1000, 3584, 3584, 1), (1000, 3584, 3588, 1), (300, 37888, 2052, 1)])
def test_the_bits_do_not_depend_on_how_groups_of_k_are_dealt_to_blocks(m, n, k, shares):
    """A row alone has a block for each group.  With a bias, and then with what is not finite in the first, a middle and the last group of some sums."""
    assert K.library().tqk_gemm_f32_shares(m, n, k) == shares
    g = torch.Generator(device="cuda").manual_seed(m + k)
    x, w = torch.randn((m, k), device="cuda", generator=g), torch.randn((n, k), device="cuda", generator=g) * 0.02
    b = torch.randn((n,), device="cuda", generator=g)
    rows = [0, 1, m // 2, m - 1]
    clean = product(x, w, b)
    for r in rows:
        assert torch.equal(product(x[r:r + 1].contiguous(), w, b)[0], clean[r]), r
    x[1, 5], x[m // 2, k // 2], x[m - 1, k - 1] = float("inf"), float("nan"), float("-inf")
    w[7, 9], w[n - 1, k - 3] = float("nan"), float("inf")
    x[3, :4], w[8, :4] = 2e19, 2e19                       # (a sum that overflows in the first group)
    y = product(x, w, b)
    for r in rows + [3]:
        one = product(x[r:r + 1].contiguous(), w, b)[0]
        assert torch.equal(one.isnan(), y[r].isnan()) and torch.equal(one.nan_to_num(), y[r].nan_to_num()), r
    finite = torch.ones((m, n), dtype=torch.bool, device="cuda")
    finite[:, [7, n - 1]], finite[[1, 3, m // 2, m - 1]] = False, False
    finite[:, 8] = False
    assert torch.equal(y[finite], clean[finite]) and torch.isinf(y[3, 8]) and not torch.isfinite(y[[1, m // 2, m - 1]]).any()


@pytest.mark.parametrize("n,k", [(1024, 1024), (1030, 1088), (2049, 516), (5003, 1028), (700, 18944)])
def test_weights_read_once_give_the_same_bits(n, k):
    """The other kind of loads: every kernel for few rows, whole stages of K and not, features that are no whole tiles; with what is not finite."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w, b = torch.randn((17, k), device="cuda", generator=g), torch.randn((n, k), device="cuda", generator=g), torch.randn((n,), device="cuda", generator=g)
    w[3, 7], x[2, k - 1] = float("inf"), float("nan")
    for m in [1, 3, 4, 5, 8, 9, 12, 16, 17]:
        for bias in (None, b):
            y = torch.full((m + 1, n), float("nan"), device="cuda")
            K.gemm(x[:m].contiguous(), w, bias, y[:m], once=True)
            want = product(x[:m].contiguous(), w, bias)
            assert y[m].isnan().all() and torch.equal(y[:m].isnan(), want.isnan()) and torch.equal(y[:m].nan_to_num(), want.nan_to_num()), m
