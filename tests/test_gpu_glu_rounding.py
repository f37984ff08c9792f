"""Gated activations in half precision: the product of two fp32 factors is rounded once, whichever kernel forms it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def product_rounded_once(a, b):
    # 24 x 24 bits fit a double, and numpy rounds a double to half precision in one step
    return torch.from_numpy((a.double().cpu().numpy() * b.double().cpu().numpy()).astype(np.float16))


@pytest.mark.parametrize("T,d", [(512, 1024), (512, 1023)])            # whole 16-byte vectors, and not
def test_gelu_times_up(T, d):
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(T, 2 * d, generator=g, device=DEV).half()
    act = _native.gelu_tanh_and_mul(torch.cat([x[:, :d].float(), torch.ones(T, d, device=DEV)], 1))       # fp32, its factor 1
    assert torch.equal(_native.gelu_tanh_and_mul(x).cpu(), product_rounded_once(act, x[:, d:].float()))


def test_clamped_glu():
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(1)
    P, ff = 512, 1024
    gu = torch.randn(P, 2 * ff, generator=g, device=DEV).half().clamp(-6, 6)
    act = _native.moe_glu(torch.cat([gu[:, :ff].float(), torch.zeros(P, ff, device=DEV)], 1), 7.0, 1.702)
    assert torch.equal(_native.moe_glu(gu, 7.0, 1.702).cpu(), product_rounded_once(act, gu[:, ff:].float() + 1.0))


def over_one_plus_exp(n, z):
    """n / (1 + exp(-z)) as the gates of every kernel form it: the fp32 head product of one column, x = 1, weight n, gate z"""
    from scratchpad_amd import _native
    one = torch.ones(1, 1, 1, device=DEV)
    return _native.head_linear(one, n.float().view(1, -1, 1).contiguous().to(DEV), z.float().view(1, -1).contiguous().to(DEV)).view(-1).cpu()


@pytest.mark.parametrize("lo,hi", [(-4.0, 4.0), (-30.0, 30.0), (-88.6, -60.0), (60.0, 120.0)])
@pytest.mark.parametrize("numerator", ["itself", "one", "2^-8 .. 2^8", "2^-90 .. 2^120"])
def test_gates_against_64_bits(numerator, lo, hi):
    """The exponential is within 2 * 2^-23 of its value, the sum behind it and the quotient add half a rounding each: 3 * 2^-23 of the result, and
    two steps of the denormals below 2^-126."""
    g = torch.Generator().manual_seed(5)
    z = lo + (hi - lo) * torch.rand(1 << 18, generator=g)
    if numerator == "itself":
        n = z
    elif numerator == "one":
        n = torch.ones_like(z)
    else:
        a, b = (-8, 8) if "8 .. " in numerator else (-90, 120)
        n = torch.exp2(a + (b - a) * torch.rand(len(z), generator=g)) * torch.where(torch.rand(len(z), generator=g) < 0.5, 1.0, -1.0)
    want = n.double() / (1 + torch.exp(-z.double()))
    assert ((over_one_plus_exp(n, z).double() - want).abs() <= 3 * 2.0 ** -23 * want.abs() + 2 * 2.0 ** -149).all()


def test_gates_at_their_ends():
    """infinities, NaN, zeros and denominators past the largest float: what n / (1 + exp(-z)) is with every operation rounded to fp32"""
    inf, nan = float("inf"), float("nan")
    n = torch.tensor([0.0, 1.0, -1.0, 2.0 ** -130, 2.0 ** 127, 3.4e38, -3.4e38, inf, -inf, nan])
    z = torch.tensor([inf, -inf, nan, 0.0, 1e-40, 17.0, 104.0, 1e5, 3.4e38, -104.0, -89.0, -1e5, -3.4e38])
    n, z = (t.reshape(-1) for t in torch.meshgrid(n, z, indexing="ij"))
    got, want = over_one_plus_exp(n, z), n / (1 + torch.exp(-z))
    assert torch.equal(got.isnan(), want.isnan())
    exact = ~want.isnan() & ((want == 0) | want.isinf() | (z >= 17) | (z.abs() < 1))          # (1 + exp(-z) is a power of two or past all floats)
    assert exact.sum() >= 90 and torch.equal(got[exact], want[exact])
    assert (got[~want.isnan()].sign() == want[~want.isnan()].sign()).all()
