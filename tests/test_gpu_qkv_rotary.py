"""sp_qkv_rotary_store where it takes a wave per token and 16-byte pieces (prompt steps without biases) and at the edges of that rule, against the
rotation in 64 bits: bf16 results of fp32 products, so half an ulp of the result and of the two terms it is the difference of."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,G,D,dims,adjacent,bias,pad", [
    (65, 4, 1, 128, 64, False, False, 0), (64, 4, 1, 128, 64, False, False, 0), (70, 3, 3, 64, 64, False, False, 0),
    (70, 2, 1, 128, 16, False, False, 0), (70, 2, 1, 128, 24, False, False, 0), (70, 2, 2, 64, 0, False, False, 0),
    (70, 4, 1, 128, 64, True, False, 0), (70, 4, 1, 128, 64, False, True, 0), (70, 4, 1, 128, 64, False, False, 4),
    (70, 2, 9, 64, 32, False, False, 0), (200, 3, 5, 32, 16, False, False, 0),
    (300, 2, 1, 320, 288, False, False, 0)])
def test_qkv_rotary_store(T, H, G, D, dims, adjacent, bias, pad, dtype):
    from scratchpad_amd import _native
    print("qkv rotary store", T, H, G, D, dims, adjacent, bias, pad, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(11)
    rn = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    a = rn(T, (H + 2 * G) * D + pad).to(dtype)
    q, k, v = a[:, :H * D], a[:, H * D:(H + G) * D], a[:, (H + G) * D:(H + 2 * G) * D]
    kp, vp = (torch.full((T + 3, G * D), float("nan"), device=DEV, dtype=dtype) for _ in range(2))
    pos, loc = torch.randint(0, 5000, (T,), generator=g, device=DEV), torch.randperm(T, generator=g, device=DEV) + 2
    freq = 10000.0 ** (-torch.arange(max(dims // 2, 1), device=DEV) / max(dims // 2, 1)) if dims else None
    biases = [rn(n * D) for n in (H, G, G)] if bias else [None] * 3
    src = [x.double() + (b.double() if b is not None else 0) for x, b in zip((q.clone(), k.clone(), v.clone()), biases)]

    def turn(x, heads):
        x = x.view(T, heads, D)
        if not dims:
            return x, x.abs()
        ang = (pos.float()[:, None] * freq).double()[:, None]
        first, second = (slice(0, dims, 2), slice(1, dims, 2)) if adjacent else (slice(0, dims // 2), slice(dims // 2, dims))
        y, size = x.clone(), x.abs()
        y[..., first] = x[..., first] * torch.cos(ang) - x[..., second] * torch.sin(ang)
        y[..., second] = x[..., second] * torch.cos(ang) + x[..., first] * torch.sin(ang)
        size[..., first] = size[..., second] = x[..., first].abs() + x[..., second].abs()
        return y, size
    _native.qkv_rotary_store(q, k, v, kp, vp, pos, loc, freq, 1.0, H, G, D, D, 1e-5, adjacent=adjacent, q_bias=biases[0],
                             k_bias=biases[1], v_bias=biases[2])
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[dtype]
    for got, x, heads in ((q, src[0], H), (kp[loc], src[1], G)):
        want, size = turn(x, heads)
        # (fp32: two products, and the angle's own cosine and sine to an ulp each)
        assert ((got.double().view(T, heads, D) - want).abs() <= half * want.abs() + 2.0 ** -21 * size).all()
    vv = src[2].view(T, G, D)
    want = (vv / torch.sqrt((vv * vv).mean(-1, keepdim=True) + 1e-5)).view(T, -1)
    assert ((vp[loc].double() - want).abs() <= half * want.abs() + 1e-5 * want.abs().max()).all()
    assert torch.isnan(kp[:2]).all() and torch.isnan(vp[:2]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,G,D,dims", [(65, 4, 1, 128, 64), (300, 3, 5, 64, 64), (70, 2, 9, 64, 32), (200, 3, 5, 32, 16), (130, 2, 1, 128, 0),
                                         (1500, 4, 4, 128, 64)])
def test_a_tokens_rows_do_not_depend_on_the_steps_size(T, H, G, D, dims, dtype):
    """the bits of a step of T tokens are those of the same tokens in steps of at most 64"""
    from scratchpad_amd import _native
    print("qkv rotary store, step sizes", T, H, G, D, dims, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(12)
    rows = torch.randn(T, (H + 2 * G) * D, generator=g, device=DEV).to(dtype)
    pos, loc = torch.randint(0, 5000, (T,), generator=g, device=DEV), torch.randperm(T, generator=g, device=DEV)
    freq = 10000.0 ** (-torch.arange(dims // 2, device=DEV) / (dims // 2)) if dims else None
    results = []
    for step in (T, 64):
        a, kp, vp = rows.clone(), *(torch.full((T, G * D), float("nan"), device=DEV, dtype=dtype) for _ in range(2))
        q, k, v = a.split([H * D, G * D, G * D], 1)
        for t0 in range(0, T, step):
            at = slice(t0, t0 + step)
            _native.qkv_rotary_store(q[at], k[at], v[at], kp, vp, pos[at], loc[at], freq, 1.0, H, G, D, D, 1e-5)
        results.append((q, kp, vp))
    for whole, parts in zip(*results):
        assert torch.isfinite(whole).all() and torch.equal(whole, parts)
