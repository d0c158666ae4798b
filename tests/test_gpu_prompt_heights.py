"""The gated product for prompts of 129 to 256 rows in blocks of five or ten waves (csrc/prompt_product.hip), at the edges of every height: the
tile the rule takes, and the result against 64 bits."""
import pytest
import torch

from tq_kv_amd import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [129, 160, 161, 192, 193, 240, 241, 255, 256])
@pytest.mark.parametrize("inter,k", [(18944, 512), (18912, 768)])
def test_gated_product_of_every_height(m, inter, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn((m, k), device="cuda", generator=g).bfloat16()
    w = (torch.randn((2 * inter, k), device="cuda", generator=g) * 0.05).bfloat16()
    assert K.prompt_tile(m, 2 * inter, k, True) == 9
    out = torch.full((m + 1, inter), float("nan"), dtype=torch.bfloat16, device="cuda")
    K.prompt_gated(x, K.pack_weight(w, 2), out[:m])
    assert torch.isnan(out[m].float()).all()
    gate, up = (x.double() @ w.double().t()).chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    # gate and up are rounded to bfloat16 (2^-9 of each, or a whole step of 2^-8 where the float32 sum falls on the other side), then the result: the derivative of
    # silu is at most silu / g + |silu|; the float32 sums are off by 2^-22 of the sum of their terms' sizes, where it is at most 1.1
    sums_g, sums_u = (2.0 ** -22 * (x.double().abs() @ w.double().abs().t())).chunk(2, 1)
    bound = 2.0 ** -8 * (want.abs() * (2.5 + gate.abs())) + 1e-4 + 1.1 * sums_g * up.abs() + sums_u * torch.nn.functional.silu(gate).abs()
    assert ((out[:m].double() - want).abs() <= bound).all()
