"""Row kernels of prompt steps at the edges of their runs and vectors, against plain torch: the request of a token row, block means
(blocks that end inside and across workgroups, widths without whole vectors), the norm of gated parts, the short convolution over
runs that cross requests."""
import pytest
import torch

from tests.test_gpu_toredra_kernels import DEV, announce, close, rms, seq_extend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1], [3, 1, 5], [255, 1, 257], [2, 0, 3, 0, 0, 700]])
def test_token_requests(lens):
    from scratchpad_amd import _native
    starts = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32, device=DEV)
    want = torch.repeat_interleave(torch.arange(len(lens)), torch.tensor(lens)).to(torch.int32)
    assert torch.equal(_native.token_requests(starts, sum(lens)).cpu(), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("P", [1, 3, 16, 17, 64])
@pytest.mark.parametrize("kw,vw", [(64, 128), (24, 40), (7, 9), (2048, 2064)])
def test_pool_blocks(P, kw, vw, dtype):
    from scratchpad_amd import _native
    announce("pool_blocks", dtype, P, kw, vw)
    g = torch.Generator(device=DEV).manual_seed(0)
    lens, prefixes, slots = [70, 1, 16, 33], [0, 2 * P + P - 1, 5, 130], [1, 2, 3, 5]
    total = sum(lens) + sum(prefixes)
    table = torch.zeros(6, 400, dtype=torch.int32, device=DEV)
    perm, at = torch.randperm(total, generator=g, device=DEV) + 1, 0
    for n, p, s in zip(lens, prefixes, slots):
        table[s, :n + p] = perm[at:at + n + p].to(torch.int32)
        at += n + p
    k, v = (torch.randn(total + 1, w, generator=g, device=DEV).to(dtype) for w in (kw, vw))
    kp, vp = torch.full_like(k, float("nan")), torch.full_like(v, float("nan"))
    _native.pool_blocks(kp, vp, k, v, table, seq_extend(lens, prefixes, slots), P)
    written = torch.zeros(total + 1, dtype=torch.bool, device=DEV)
    for n, p, s in zip(lens, prefixes, slots):
        for pos in range(p, p + n):
            if (pos + 1) % P == 0:
                rows, dst = table[s, pos - P + 1:pos + 1].long(), int(table[s, pos])
                written[dst] = True
                for got, src in ((kp, k), (vp, v)):
                    want = src[rows].double().mean(0)
                    bar = 2.0 ** -8 if dtype == torch.bfloat16 else (P + 2) * 2.0 ** -23
                    assert ((got[dst].double() - want).abs() <= bar * src[rows].double().abs().mean(0) + 1e-30).all()
    assert torch.isnan(kp[~written]).all() and torch.isnan(vp[~written]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("P", [16, 31, 33, 50, 64, 65, 130, 257])
@pytest.mark.parametrize("kw,vw", [(64, 128), (256, 256), (256, 264), (512, 512), (520, 504), (512, 520), (7, 9)])
def test_pool_blocks_add_their_rows_in_order(P, kw, vw, dtype):
    """whole, half and quarter pieces per thread, partial rounds and more rows than lanes: the bits of the rows added one after the
    other in fp32, whatever the width - a block's mean does not depend on what else the kernel is launched for"""
    from scratchpad_amd import _native
    announce("pool_blocks in order", dtype, P, kw, vw)
    g = torch.Generator(device=DEV).manual_seed(3)
    lens, prefixes, slots = [1, P + 3, 2 * P, 1], [P - 1, 5, 0, 3 * P - 1], [1, 2, 3, 5]
    total = sum(lens) + sum(prefixes)
    table = torch.zeros(6, 4 * P + 8, dtype=torch.int32, device=DEV)
    perm, at = torch.randperm(total, generator=g, device=DEV) + 1, 0
    for n, p, s in zip(lens, prefixes, slots):
        table[s, :n + p] = perm[at:at + n + p].to(torch.int32)
        at += n + p
    k, v = (torch.randn(total + 1, w, generator=g, device=DEV).to(dtype) for w in (kw, vw))
    kp, vp = torch.full_like(k, float("nan")), torch.full_like(v, float("nan"))
    _native.pool_blocks(kp, vp, k, v, table, seq_extend(lens, prefixes, slots), P)
    ends = [(table[s, pos - P + 1:pos + 1].long(), int(table[s, pos])) for n, p, s in zip(lens, prefixes, slots)
            for pos in range(p, p + n) if (pos + 1) % P == 0]
    rows, dst = torch.stack([r for r, _ in ends]), torch.tensor([d for _, d in ends], device=DEV)
    for got, src in ((kp, k), (vp, v)):
        acc = torch.zeros(len(ends), src.shape[1], device=DEV)
        for j in range(P):
            acc += src[rows[:, j]].float()
        inv = (torch.tensor(1.0) / P).to(DEV)
        same = got[dst] == (acc * inv).to(dtype)
        if dtype == torch.float16:      # (an instruction multiplies in 32 bits and rounds once, to 16; numpy's cast does so from 64)
            once = (acc.double() * inv.double()).cpu().numpy().astype("float16")
            same |= got[dst] == torch.from_numpy(once).to(DEV)
        assert same.all()
        assert int(torch.isnan(got).any(1).sum()) == total + 1 - len(ends)


@pytest.mark.parametrize("B", [1, 17, 256, 257])
def test_pool_blocks_of_requests_that_complete_together(B):
    """decode steps whose requests all end a block, on both sides of the line between one row and sixteen per workgroup"""
    from scratchpad_amd import _native
    announce("pool_blocks together", B)
    g = torch.Generator(device=DEV).manual_seed(21)
    P, W = 16, 64
    table = (torch.randperm(B * P, generator=g, device=DEV) + 1).to(torch.int32).view(B, P)
    table = torch.cat([torch.zeros(1, P, dtype=torch.int32, device=DEV), table])
    k, v = (torch.randn(B * P + 1, W, generator=g, device=DEV).bfloat16() for _ in range(2))
    kp, vp = torch.full_like(k, float("nan")), torch.full_like(v, float("nan"))
    seq = _native.SeqParams(torch.arange(1, B + 1, device=DEV), torch.full((B,), P, device=DEV))
    _native.pool_blocks(kp, vp, k, v, table, seq, P)
    rows = table[1:].long()
    for got, src in ((kp, k), (vp, v)):
        want = src[rows].double().mean(1)
        assert ((got[rows[:, -1]].double() - want).abs() <= 2.0 ** -8 * src[rows].double().abs().mean(1)).all()
        assert int(torch.isnan(got).all(1).sum()) == B * P + 1 - B


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,parts,per", [(1, 1, 8), (5, 3, 512), (3, 2, 520), (7, 1, 1024), (2, 3, 2048), (2, 1, 2056), (3, 4, 37)])
def test_gated_group_norm(T, parts, per, dtype):
    from scratchpad_amd import _native
    announce("gated_group_norm", dtype, T, parts, per)
    g = torch.Generator(device=DEV).manual_seed(1)
    n = parts * per
    y, w = torch.randn(T, n, generator=g, device=DEV), torch.rand(n, generator=g, device=DEV) + 0.5
    z = (torch.randn(T, n + 64, generator=g, device=DEV) * 4).to(dtype)[:, :n]
    z[0, 0] = -100.0
    v = y.double() * torch.nn.functional.silu(z.double())
    want = (rms(v.view(T, parts, per), 1e-5).view(T, n) * w.double()).double()
    got = _native.gated_group_norm(y, z, w, parts, 1e-5).double()
    bar = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10, torch.float32: 1e-5}[dtype]
    assert ((got - want).abs() <= bar * want.abs() + 1e-6).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("C", [8, 264, 2056])
@pytest.mark.parametrize("lens,prefixes", [([8], [0]), ([16, 9, 1, 22], [0, 2, 7, 0]), ([40], [1]), ([7, 8, 8, 1], [3, 0, 5, 1])])
@pytest.mark.parametrize("taps", [2, 4])
def test_causal_conv_runs(lens, prefixes, C, taps, dtype):
    from scratchpad_amd import _native
    announce("conv", dtype, lens, prefixes, C, taps)
    g = torch.Generator(device=DEV).manual_seed(2)
    T, slots = sum(lens), list(range(1, len(lens) + 1))
    x = torch.randn(T, C + 8, generator=g, device=DEV).to(dtype)[:, :C]
    w, bias = torch.randn(C, taps, generator=g, device=DEV), torch.randn(C, generator=g, device=DEV)
    state = torch.randn(len(lens) + 1, taps - 1, C, generator=g, device=DEV)
    before, at, want = state.clone(), 0, []
    for n, p, s in zip(lens, prefixes, slots):
        past = before[s].double().clone()
        past[:max(0, taps - 1 - p)] = 0                            # entries before the sequence's start are not read
        pad = torch.cat([past, x[at:at + n].double()])
        want.append(torch.nn.functional.silu(sum(pad[j:j + n] * w[:, j].double() for j in range(taps)) + bias.double()))
        at += n
    got = _native.causal_conv_silu(x, w, bias, state, seq_extend(lens, prefixes, slots))
    want = torch.cat(want)
    bar = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-5
    # (a silu near its zero takes the absolute error of the sum before it)
    assert ((got.double() - want).abs() <= bar * want.abs() + 4e-6).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", [[65], [3, 1, 1, 60, 16, 17, 2], [1] * 70, [5000, 9, 3190]], ids=lambda l: str(sum(l)))
@pytest.mark.parametrize("C,taps", [(8, 4), (264, 3), (1032, 2), (16, 1)])
def test_causal_conv_of_long_steps(lens, C, taps, dtype):
    """runs of 8 and of 16 tokens in which requests end, the last one short; fewer pieces of a row than lanes"""
    from scratchpad_amd import _native
    announce("conv", dtype, lens[:8], len(lens), C, taps)
    g = torch.Generator(device=DEV).manual_seed(4)
    prefixes, slots = [(0, 2, 7)[i % 3] for i in range(len(lens))], list(range(1, len(lens) + 1))
    x = torch.randn(sum(lens), C + 8, generator=g, device=DEV).to(dtype)[:, 8:]
    w, bias = torch.randn(C, taps, generator=g, device=DEV), torch.randn(C, generator=g, device=DEV)
    state = torch.randn(len(lens) + 1, taps - 1, C, generator=g, device=DEV)
    before, at, want = state.clone(), 0, []
    for n, p, s in zip(lens, prefixes, slots):
        past = before[s].double().clone()
        past[:max(0, taps - 1 - p)] = 0
        pad = torch.cat([past, x[at:at + n].double()])
        want.append(torch.nn.functional.silu(sum(pad[j:j + n] * w[:, j].double() for j in range(taps)) + bias.double()))
        at += n
    got = _native.causal_conv_silu(x, w, bias, state, seq_extend(lens, prefixes, slots))
    want = torch.cat(want)
    bar = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 1e-5}[dtype]          # as in test_causal_conv_runs
    assert ((got.double() - want).abs() <= bar * want.abs() + 4e-6).all()


@pytest.mark.parametrize("T", [65, 96, 257])
@pytest.mark.parametrize("K,n,bias", [(32, 1, True), (288, 16, False), (2048, 31, True), (1024, 64, False), (544, 131, True)])
def test_fp32_products_of_many_rows(T, K, n, bias):
    """fp32 weights of all magnitudes against 64 bits: K fp32 additions and roundings of exact products"""
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(T + K + n)
    wide = torch.randn(T, K + 8, generator=g, device=DEV).bfloat16()
    x = wide[:, 8:]                                                       # a view, 16-byte aligned rows
    w = torch.randn(n, K, generator=g, device=DEV) * torch.exp2(torch.randint(-30, 31, (n, 1), generator=g, device=DEV).float())
    b = torch.randn(n, generator=g, device=DEV) if bias else None
    out = _native.small_linear_f32(x, w, b)
    want = x.double() @ w.double().T + (b.double() if bias else 0.0)
    bound = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + (b.double().abs() if bias else 0.0))
    assert out.shape == (T, n) and bool(((out.double() - want).abs() <= bound).all())


# tiles of 64 rows, the last of few; of 32 rows again; few rows of a long K and of many outputs
@pytest.mark.parametrize("T,K,n", [(2100, 1056, 64), (4097, 96, 17), (8193, 64, 16), (100, 16384, 40), (71, 4096, 2050)])
def test_fp32_products_of_more_rows(T, K, n):
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(T + K + n)
    x = torch.randn(T, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(n, K, generator=g, device=DEV)
    out = _native.small_linear_f32(x, w)
    bound = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((out.double() - x.double() @ w.double().T).abs() <= bound).all())
    few = _native.small_linear_f32(x[T - 70:], w)                     # the order of a row's sum is K's alone
    assert torch.equal(out[T - 70:], few)


# tiles of 64 rows: the widest stride that they take, the first past 32 bits; the same of 32
@pytest.mark.parametrize("stride,n", [(1 << 25, 1376), (34087048, 1376), (1 << 26, 16), (69273672, 16)])
def test_fp32_products_of_far_apart_rows(stride, n):
    """the entry and its wrapper take rows any distance apart"""
    from scratchpad_amd import _native
    T, K = 65, 64
    announce("fp32 products of far rows", stride, n)
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.empty(stride * (T - 1) + K, dtype=torch.bfloat16, device=DEV).as_strided((T, K), (stride, 1))
    x.copy_(torch.randn(T, K, generator=g, device=DEV))
    w = torch.randn(n, K, generator=g, device=DEV)
    want, bound = x.double() @ w.double().T, (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    out = torch.empty(T, n, device=DEV)
    _native._check(_native.load().sp_small_linear_f32(out.data_ptr(), x.data_ptr(), stride, w.data_ptr(), None, T, K, n, _native._dt(x),
                                                      _native._stream()), "sp_small_linear_f32")
    for got in (out, _native.small_linear_f32(x, w)):
        assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("T", [64, 65, 100])
def test_fp32_products_of_infinite_inputs(T):
    """an infinity is one in the sum it enters, in every form: not NaN"""
    from scratchpad_amd import _native
    K, n = 96, 20
    x, w = torch.ones(T, K, device=DEV).bfloat16(), torch.full((n, K), 0.5, device=DEV)
    x[3, 5], x[60, 95], x[9, 0] = float("inf"), float("-inf"), float("nan")
    w[7, 31], w[8, 2] = float("inf"), 1.1                             # (1.1: a weight of three parts)
    want = torch.nn.functional.linear(x.cpu().double(), w.cpu().double())
    got = _native.small_linear_f32(x, w).cpu().double()
    assert torch.isnan(want[9]).all() and torch.isinf(want[3]).all() and torch.isnan(want[60, 7])
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.allclose(got, want, rtol=1e-5, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_of_every_16_bit_value(dtype):
    """the convolution's SiLU of every number of the type: its one rounding and little else"""
    from scratchpad_amd import _native
    C, T = 1024, 64
    x = torch.arange(65536, dtype=torch.int32, device=DEV).to(torch.int16).view(dtype).view(T, C).clone()
    x[~torch.isfinite(x)] = 0.0
    w = torch.zeros(C, 4, device=DEV)
    w[:, 3] = 1.0
    got = _native.causal_conv_silu(x, w, None, torch.zeros(2, 3, C, device=DEV), seq_extend([T], [0], [1])).double()
    want = x.double() * torch.sigmoid(x.double())
    half = torch.exp2(torch.frexp(want)[1].double() - 1 - (8 if dtype == torch.bfloat16 else 11))          # half a step at the result
    # what fp32 adds: four roundings.  Its exponential ends at e^88.72: below -88.72 the result is zero, 2.7e-37 off; subnormal halves
    # keep 2^-25
    floor = 3e-37 if dtype == torch.bfloat16 else 2.0 ** -25
    assert ((got - want).abs() <= half + 2.0 ** -22 * want.abs() + floor).all()

@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(300, 2048), (300, 2056), (300, 4096), (257, 8192), (2049, 6144)])
def test_rmsnorm_of_many_rows_is_that_of_a_few(rows, hidden, dtype):
    """where the loads are issued depends on type, rows and width, a row's bits do not: many rows at once against 128 at a time"""
    from scratchpad_amd import _native
    announce("rmsnorm", dtype, rows, hidden)
    g = torch.Generator().manual_seed(rows + hidden)
    x, res, w = (torch.randn(*s, generator=g).to(dtype).to(DEV) for s in ((rows, hidden), (rows, hidden), (hidden,)))
    parts = [slice(i, min(i + 128, rows)) for i in range(0, rows, 128)]
    many = _native.rmsnorm(x, w, 1e-5)
    assert torch.equal(many, torch.cat([_native.rmsnorm(x[p], w, 1e-5) for p in parts]))
    few_x, few_res = x.clone(), res.clone()
    for p in parts:
        _native.fused_add_rmsnorm(few_x[p], few_res[p], w, 1e-5)
    _native.fused_add_rmsnorm(x, res, w, 1e-5)
    assert torch.equal(x, few_x) and torch.equal(res, few_res)
