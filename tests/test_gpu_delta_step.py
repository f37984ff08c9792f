"""sp_delta_step (a decode step of the generalized delta rule, its gates formed inside) against sp_delta_gates followed by
sp_delta_recurrence: the same fp32 sums in other orders, so the states differ by fp32 roundings of sums of 64 to 512 products and
the outputs by those and one rounding of their type."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bar", [(torch.bfloat16, 2.0 ** -7), (torch.float16, 2.0 ** -10), (torch.float32, 1e-4)])
@pytest.mark.parametrize("B,H,D,rank", [(1, 1, 64, 64), (3, 5, 64, 1), (16, 16, 64, 64), (2, 3, 128, 96), (5, 2, 64, 512)])
def test_step_against_gates_and_recurrence(dtype, bar, B, H, D, rank):
    from scratchpad_amd import _native
    g = torch.Generator(device="cuda").manual_seed(B * 100 + H + rank)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    n = H * D
    a = rnd(B, 5 * n + rank).to(dtype)                                   # views of one product
    r, k, v, gt, ap, p = a.split([n, n, n, n, n, rank], 1)
    w2t, w0, ab, nw = rnd(rank, n) * rank ** -0.5, rnd(n), rnd(n), torch.rand(n, generator=g, device="cuda") + 0.5
    slots = torch.arange(B, device="cuda") * 2 + 1
    lens = torch.tensor([1 if i == 1 else 5 + i for i in range(B)], device="cuda")      # request 1 starts with this token
    seq = _native.SeqParams(slots, lens)
    S = torch.full((2 * B + 1, H, D, D), float("nan"), device="cuda")
    S[slots] = rnd(B, H, D, D)
    S2 = S.clone()
    got = _native.delta_step(r, k, v, gt, p, ap, w2t, w0, ab, 0.6, nw, S, seq, H, D, 1e-5)
    dec, rem = _native.delta_gates(p, w2t, w0, ap, ab, 0.6)
    want = _native.delta_recurrence(r, k, v, gt, dec, rem, nw, S2, seq, H, D, 1e-5)
    assert float((S[slots] - S2[slots]).abs().max()) <= 2e-5 * float(S2[slots].abs().max())
    assert bool((got.double() - want.double()).abs().le(bar * want.double().abs() + 1e-4).all())
    others = torch.ones(2 * B + 1, dtype=torch.bool, device="cuda")
    others[slots] = False
    assert torch.isnan(S[others]).all()                                  # no state but the requests' own


def test_step_takes_other_forms_as_two_launches():
    from scratchpad_amd import _native
    torch.manual_seed(3)
    B, H, D, rank = 2, 3, 16, 8                                          # heads of 16
    n = H * D
    r, k, v, gt, ap, p = torch.randn(B, 5 * n + rank, device="cuda").split([n, n, n, n, n, rank], 1)
    w2t, w0, ab, nw = torch.randn(rank, n, device="cuda"), *(torch.randn(n, device="cuda") for _ in range(3))
    seq = _native.SeqParams(torch.tensor([1, 2], device="cuda"), torch.tensor([4, 9], device="cuda"))
    S = torch.randn(3, H, D, D, device="cuda")
    S2 = S.clone()
    got = _native.delta_step(r, k, v, gt, p, ap, w2t, w0, ab, 0.6, nw, S, seq, H, D, 1e-5)
    dec, rem = _native.delta_gates(p, w2t, w0, ap, ab, 0.6)
    want = _native.delta_recurrence(r, k, v, gt, dec, rem, nw, S2, seq, H, D, 1e-5)
    assert torch.equal(got, want) and torch.equal(S, S2)
