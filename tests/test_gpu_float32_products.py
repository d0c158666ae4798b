"""float32 products with large weights, whose numbers go through the matrix cores as three bfloat16 ones each (csrc/gemm_generic.hip): the
same bits whatever the number of rows (one kernel each for up to 4, 8 and 16 rows, four tiles for more), and no further from 64 bits than float32
sums are; infinities, NaN and numbers that overflow come out as float32 arithmetic gives them."""
import pytest
import torch

from tq_kv_amd import kernels as K

pytestmark = pytest.mark.gpu
ROWS = [1, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 130]


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
    # A float32 sum by chunks: within a chunk each of four instructions' sums of 32 k and five small ones rounds once, 24 roundings of a sum that grows to the chunk's size, and one
    # for each of the chunks, groups and the bias, 2^-24 of what is summed so far each and independent: no more than sqrt(24 / 3 + 2) 2^-24 of the result's spread, and the same
    # again for terms that cancel.
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
