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
