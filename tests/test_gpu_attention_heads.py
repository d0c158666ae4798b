"""Heads of a kv head together in the generic attention kernel (csrc/attention_generic.hip): the bits of the general kernel, over groups, head sizes,
counts of queries, windows and tables on both sides of each line of its rule."""
import pytest
import torch

from tq_kv_amd import kernels as K

pytestmark = pytest.mark.gpu
SPARE = 8               # page table columns that no query reaches (tables may be wider than the sequences)


@pytest.mark.parametrize("nh,nkv", [(2, 1), (6, 2), (28, 4), (9, 1), (17, 1)])
@pytest.mark.parametrize("d", [4, 20, 64, 100, 128])
@pytest.mark.parametrize("window", [0, 70, 600])
def test_heads_together_give_the_general_kernels_bits(nh, nkv, d, window):
    g = torch.Generator(device="cuda").manual_seed(nh * d + window)
    n_pages = 12
    keys = torch.randn((n_pages + 1, nkv, 64, d), device="cuda", generator=g)
    values = torch.randn((n_pages + 1, nkv, d, 64), device="cuda", generator=g)
    order = torch.randperm(n_pages, generator=torch.Generator().manual_seed(d))
    wide = torch.full((2, n_pages + SPARE), -1, dtype=torch.int32)
    wide[0, :n_pages], wide[1, 0] = order.int(), n_pages                # a second sequence of one page
    edges = torch.tensor([0, 1, 62, 63, 64, 65, 69, 70, 127, 128, 200, 255])
    longer = torch.tensor([256, 300, 511, 512, 599, 600, 601, 700, 767])
    for some, pages in ((edges, 4), (torch.cat([edges, longer]), n_pages + SPARE)):
        table = wide[:, :pages].contiguous().cuda()
        for n in (256 // nh + 1, 512 // nh + 1, 2000 // nh + 1):
            pos = some[torch.arange(n) % len(some)].int()
            seq = (torch.arange(n) % 7 == 3).int()
            pos = torch.where(seq == 1, pos % 64, pos).int().cuda()
            seq = seq.cuda()
            q = torch.randn((n, nh, d), device="cuda", generator=g)
            out = torch.full((n + 1, nh * d), float("nan"), device="cuda")
            K.attention(q, keys, values, seq, pos, table, window, d ** -0.5, out[:n])
            assert torch.isnan(out[n]).all()
            few = torch.empty((n, nh * d), device="cuda")               # no more than 256 waves of queries: the general kernel
            step = 256 // nh
            for i in range(0, n, step):
                part = slice(i, min(n, i + step))
                K.attention(q[part], keys, values, seq[part], pos[part], table, window, d ** -0.5, few[part])
            assert torch.equal(out[:n], few), (n, pages)


def test_scores_of_minus_infinity_and_infinities_in_values():
    """Whole pages of scores -inf, and values that are infinite in positions a query does not see."""
    nh, nkv, d, n = 8, 2, 64, 80
    g = torch.Generator(device="cuda").manual_seed(5)
    keys, values = torch.randn((4, nkv, 64, d), device="cuda", generator=g), torch.randn((4, nkv, d, 64), device="cuda", generator=g)
    keys[1, :, :, 0] = float("-inf")                                    # page 1: every score -inf for queries with a positive first value
    values[3] = float("inf")
    q = torch.randn((n, nh, d), device="cuda", generator=g)
    q[:, :, 0] = q[:, :, 0].abs() + 0.1
    pos = torch.full((n,), 191, dtype=torch.int32, device="cuda")
    table = torch.tensor([[1, 0, 2, 3]], dtype=torch.int32, device="cuda")
    seq = torch.zeros(n, dtype=torch.int32, device="cuda")
    out, few = torch.empty((n, nh * d), device="cuda"), torch.empty((n, nh * d), device="cuda")
    K.attention(q, keys, values, seq, pos, table, 0, d ** -0.5, out)
    for i in range(0, n, 20):
        K.attention(q[i:i + 20], keys, values, seq[i:i + 20], pos[i:i + 20], table, 0, d ** -0.5, few[i:i + 20])
    assert torch.equal(out, few) and torch.isfinite(out).all()
