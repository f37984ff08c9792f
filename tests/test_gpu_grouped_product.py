"""The grouped expert products on the matrix cores at the edges of their tiles (rows per expert around 16, 64, 128 and 320, columns
and k that end inside a tile, experts without rows, more experts than lanes), against the product in fp32 by torch, and the
gated form bit for bit against the product followed by its activation."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def grouped_inputs(counts, N, K, dtype, top, seed=0):
    """rows sorted by expert with the given counts; order holds pairs (token * top + k) in a shuffled order"""
    g = torch.Generator(device=DEV).manual_seed(seed)
    E, P = len(counts), sum(counts)
    tokens = (P + top - 1) // top
    a = torch.randn(tokens, K, generator=g, device=DEV).to(dtype)
    w = (torch.randn(E, N, K, generator=g, device=DEV) * K ** -0.5).to(dtype)
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=DEV)
    order = torch.randperm(tokens * top, generator=g, device=DEV)[:P].to(torch.int32)
    expert = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(counts, device=DEV))
    return a, w, offsets, order, expert, P


COUNTS = [[1], [0, 3, 0, 17], [16, 0, 15, 33], [63, 64, 65, 1], [127, 128, 129, 257, 0], [300, 2, 140], [3] * 70, [90] * 67 + [0, 1],
          [321], [0, 385, 700, 129], [1100] + [1] * 2,
          [2, 0, 1, 0, 1], [0] * 66 + [17, 1, 0, 40]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: "-".join(map(str, c[:5])))
@pytest.mark.parametrize("N,K", [(64, 32), (130, 96), (200, 256), (300, 160)])
def test_grouped_products(counts, N, K, dtype):
    from scratchpad_amd import _native
    top = 3
    print("grouped", counts[:6], len(counts), N, K, dtype, flush=True)
    a, w, offsets, order, expert, P = grouped_inputs(counts, N, K, dtype, top)
    # one rounding of the result plus fp32 sums: half an ulp of the 16-bit type, and K fp32 additions
    bar = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + K * 2.0 ** -23
    rows = a[(order // top).long()].float()
    want = torch.cat([rows[expert == e] @ w[e].float().t() for e in range(len(counts))])
    scale = rows.abs().max() * w.float().abs().sum(-1).max()
    for got, ref in ((_native.moe_grouped_gemm(a, w, offsets, P, order, top), want),
                     (_native.moe_grouped_gemm(a, w, offsets, P, order, top, act="relu2"), torch.relu(want) ** 2)):
        assert ((got.float() - ref).abs() <= 2 * bar * ref.abs() + K * 2.0 ** -22 * scale).all()
    plain = _native.moe_grouped_gemm(rows.to(dtype), w, offsets, P)
    assert torch.equal(plain, _native.moe_grouped_gemm(a, w, offsets, P, order, top))
    # an output row has the same bits whichever tile height computes it: alone, its expert takes the few-rows kernel
    for e in [e for e, c in enumerate(counts) if c][:3]:
        at = int(offsets[e])
        one = torch.zeros_like(offsets)
        one[e + 1:] = 1
        assert torch.equal(_native.moe_grouped_gemm(rows[at:at + 1].to(dtype), w, one, 1)[0], plain[at])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: "-".join(map(str, c[:5])))
@pytest.mark.parametrize("ff,K", [(32, 32), (67, 96), (136, 128), (260, 64)])
def test_gated_form_is_the_two_steps(counts, ff, K, dtype):
    from scratchpad_amd import _native
    a, w, offsets, order, _, P = grouped_inputs(counts, 2 * ff, K, dtype, 2, seed=1)
    print("gated", counts[:6], ff, K, dtype, flush=True)
    a = a * 3                                                     # beyond the clamp too
    gu = _native.moe_grouped_gemm(a, w, offsets, P, order, 2)
    assert torch.equal(_native.moe_grouped_glu(a, w, offsets, P, order, 2, "silu"), _native.silu_and_mul(gu))
    assert torch.equal(_native.moe_grouped_glu(a, w, offsets, P, order, 2, "clamped", 2.0, 1.702), _native.moe_glu(gu, 2.0, 1.702))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [480, 512, 544, 1024, 1056])
@pytest.mark.parametrize("E,pairs,N", [(8, 4, 512), (8, 4, 1024), (8, 4, 1028), (8, 8, 513), (16, 2, 2048), (8, 9, 256), (32, 24, 1024)])
def test_few_pairs_have_the_bits_of_many(E, pairs, N, K, dtype):
    """few pairs over whole and partial rounds of k-steps, at both sides of the line of one wave per compute unit and at one to one and a
    half per SIMD: the bits of the same rows beside so many others that another kernel takes them, in the product and in its gated form"""
    from scratchpad_amd import _native
    print("few pairs", E, pairs, N, K, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(6)
    a = torch.randn(pairs, K, generator=g, device=DEV).to(dtype)
    many = torch.randn(24 * E, K, generator=g, device=DEV).to(dtype)
    w = (torch.randn(E, 2 * N, K, generator=g, device=DEV) * K ** -0.5).to(dtype)
    expert = torch.sort(torch.randint(0, E, (pairs,), generator=g, device=DEV)).values
    counts = torch.bincount(expert, minlength=E)
    offsets = torch.cat([counts.new_zeros(1), counts.cumsum(0)]).int()
    # the same rows at the head of their experts' groups of a step of 24 more rows per expert
    big = torch.cat([torch.cat([a[expert == e], many[24 * e:24 * (e + 1)]]) for e in range(E)])
    big_offsets = (offsets + 24 * torch.arange(E + 1, device=DEV)).int()
    at = torch.arange(pairs, device=DEV) + 24 * expert
    for width in (N, 2 * N):
        ww = w[:, :width].contiguous()
        got = _native.moe_grouped_gemm(a, ww, offsets, pairs)
        want = (a.float()[:, None] * ww[expert].float()).sum(-1)
        size = (a.float()[:, None] * ww[expert].float()).abs().sum(-1)
        bar = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11          # half an ulp, and K fp32 additions in either order
        assert ((got.float() - want).abs() <= bar * want.abs() + 2 * K * 2.0 ** -24 * size).all()
        assert torch.equal(got, _native.moe_grouped_gemm(big, ww, big_offsets, big.shape[0])[at])
    for act, more in (("silu", ()), ("clamped", (2.0, 1.702))):
        got = _native.moe_grouped_glu(a, w, offsets, pairs, None, 1, act, *more)
        assert torch.equal(got, _native.moe_grouped_glu(big, w, big_offsets, big.shape[0], None, 1, act, *more)[at])


def test_gated_form_leaves_other_shapes_to_the_two_steps():
    from scratchpad_amd import _native
    for dtype, K in ((torch.float32, 64), (torch.bfloat16, 40)):
        a, w, offsets, order, _, P = grouped_inputs([2, 5], 16, K, dtype, 2)
        assert _native.moe_grouped_glu(a, w, offsets, P, order, 2, "silu") is None


def test_few_rows_of_very_many_experts():
    """more row tiles than a launch's second dimension holds"""
    from scratchpad_amd import _native
    E, N, K = 70000, 32, 32
    g = torch.Generator(device=DEV).manual_seed(3)
    a, w = (torch.randn(E, *s, generator=g, device=DEV).bfloat16() for s in ((K,), (N, K)))
    offsets = torch.arange(E + 1, dtype=torch.int32, device=DEV)
    got = _native.moe_grouped_gemm(a, w, offsets, E)
    want = (a.float()[:, None] * w.float()).sum(-1)
    assert ((got.float() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -22 * (a.float().abs()[:, None] * w.float().abs()).sum(-1)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,width,top", [(1, 8, 1), (5, 264, 4), (3, 2056, 6), (9, 37, 5)])
def test_combine(T, width, top, dtype):
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(2)
    z = torch.randn(T * top, width, generator=g, device=DEV).to(dtype)
    place = torch.randperm(T * top, generator=g, device=DEV).to(torch.int32).view(T, top)
    wt = torch.rand(T, top, generator=g, device=DEV)
    want = (z.float()[place.long()] * wt[..., None]).sum(1)
    bar = 2.0 ** -8 if dtype == torch.bfloat16 else top * 2.0 ** -23
    assert ((_native.moe_combine(z, place.view(-1), wt).float() - want).abs() <= bar * want.abs() + 1e-5).all()


# (experts, mean rows, weight rows, K): the sizes at which each of the ring kernel's ten tiles is the one taken, K of fewer steps than a ring holds and more
RING = [(2, 16, 128, 64), (8, 30, 200, 192), (2, 12, 128, 512), (2, 100, 128, 512), (32, 300, 200, 64), (32, 200, 384, 320), (16, 800, 200, 320),
        (16, 800, 384, 64), (16, 150, 1024, 192), (32, 300, 200, 256), (32, 800, 200, 64), (8, 800, 1024, 64), (32, 500, 512, 64), (8, 500, 2048, 64),
        (32, 800, 384, 64), (32, 150, 2048, 64), (16, 800, 512, 1024), (4, 800, 2048, 512),
        (2, 12, 128, 320), (2, 100, 128, 1024), (32, 40, 1000, 1024), (32, 150, 384, 1024), (2, 60, 128, 512), (32, 80, 1000, 1024),
        (32, 120, 1000, 1024), (16, 300, 1000, 1024), (32, 180, 1000, 320)]


def rows_kernel_share(E, N, K):
    """of so many pairs, among the experts and as many more without rows, the rows kernel takes both forms: their weights are no stream"""
    from scratchpad_amd import _native
    takes = lambda n: all(_native.load().sp_moe_grouped_plan(gated, 2, n, N >> gated, K, E + n, K) in (0, 1) for gated in (0, 1))          # noqa: E731
    share = max(n for n in (16, 32, 64, 128, 256, 512, 1024, 2048, 4096) if takes(n))
    assert all(takes(n) for n in range(1, share))
    return share


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,mean,N,K", RING)
def test_ring_tiles_have_the_bits_of_the_rows_kernel(E, mean, N, K, dtype):
    """the same rows a share at a time, among so many experts without any that the rows kernel takes them; uneven experts, one without rows and
    one with one"""
    from scratchpad_amd import _native
    print("ring", E, mean, N, K, dtype, flush=True)
    counts = [mean] * E
    counts[0], counts[1] = 2 * mean - 1, 1
    if E > 2:
        counts[2], counts[3] = 0, 2 * mean
    a, w, offsets, order, expert, P = grouped_inputs(counts, N, K, dtype, 2, seed=7)
    plans = [_native.load().sp_moe_grouped_plan(gated, 2, P, N >> gated, K, E, K) for gated in (0, 1)]
    assert plans[0] >= 16 and plans[1] >= (16 if mean <= 320 else 4)
    share = rows_kernel_share(E, N, K)
    many = torch.empty(E + share, N, K, dtype=dtype, device=DEV)               # (experts without rows are not read)
    many[:E] = w

    def by_rows(product):
        out = []
        for at in range(0, P, share):
            n = min(share, P - at)
            some = (offsets.clamp(at, at + n) - at).to(torch.int32)
            out.append(product(torch.cat([some, some[-1:].expand(n)]).contiguous(), many[:E + n], n, order[at:at + n]))
        return torch.cat(out)

    got = _native.moe_grouped_gemm(a, w, offsets, P, order, 2)
    assert torch.equal(got, by_rows(lambda o, m, n, rows: _native.moe_grouped_gemm(a, m, o, n, rows, 2)))
    rows = a[(order // 2).long()].float()
    want = torch.cat([rows[expert == e] @ w[e].float().t() for e in range(E)])
    scale = rows.abs().max() * w.float().abs().sum(-1).max()
    bar = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11                  # as in test_grouped_products
    assert ((got.float() - want).abs() <= 2 * bar * want.abs() + K * 2.0 ** -22 * scale).all()
    assert torch.equal(_native.moe_grouped_gemm(a, w, offsets, P, order, 2, act="relu2"),
                       by_rows(lambda o, m, n, rows: _native.moe_grouped_gemm(a, m, o, n, rows, 2, act="relu2")))
    for act in (("silu",), ("clamped", 2.0, 1.702)):
        assert torch.equal(_native.moe_grouped_glu(a, w, offsets, P, order, 2, *act),
                           by_rows(lambda o, m, n, rows: _native.moe_grouped_glu(a, m, o, n, rows, 2, *act)))


def test_rows_far_from_the_first():
    """rows of `a` that 32-bit offsets do not reach, named by an order of fewer pairs"""
    from scratchpad_amd import _native
    K, N, E, P = 4096, 64, 2, 100
    a = torch.zeros(2 ** 31 // K + P, K, dtype=torch.bfloat16, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(9)
    a[-P:] = torch.randn(P, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(E, N, K, generator=g, device=DEV) * K ** -0.5).bfloat16()
    offsets = torch.tensor([0, 40, P], dtype=torch.int32, device=DEV)
    order = torch.arange(a.shape[0] - P, a.shape[0], dtype=torch.int32, device=DEV)
    near = a[-P:].clone()
    assert torch.equal(_native.moe_grouped_gemm(a, w, offsets, P, order), _native.moe_grouped_gemm(near, w, offsets, P))
    assert torch.equal(_native.moe_grouped_glu(a, w, offsets, P, order, 1, "silu"), _native.moe_grouped_glu(near, w, offsets, P, None, 1, "silu"))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("row_div", [1, 2])
@pytest.mark.parametrize("counts", [[40, 60], [7, 0, 300, 293], [33, 1567], [70] * 16], ids=lambda c: str(sum(c)))
def test_orders_of_near_and_far_rows(counts, row_div, dtype):
    """an order names any rows: first ones, ones on either side of 2^31 elements and the last, in one row tile; the bits of the same rows gathered"""
    from scratchpad_amd import _native
    K, N, E, P = 512, 200, len(counts), sum(counts)
    print("far", counts[:4], row_div, dtype, flush=True)
    g = torch.Generator(device=DEV).manual_seed(11)
    edge = 2 ** 31 // K
    a = torch.empty(edge + 2 * P, K, dtype=dtype, device=DEV)
    rows = torch.cat([torch.arange(P, device=DEV), torch.arange(edge - P, edge + P, device=DEV), torch.arange(a.shape[0] - P, a.shape[0], device=DEV)])
    a[rows] = torch.randn(len(rows), K, generator=g, device=DEV).to(dtype)
    rows = rows[torch.randperm(len(rows), generator=g, device=DEV)[:P]]
    order = (rows * row_div + row_div - 1).to(torch.int32)
    w = (torch.randn(E, 2 * N, K, generator=g, device=DEV) * K ** -0.5).to(dtype)
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=DEV)
    near = a[rows].clone()
    for act in ("none", "relu2"):
        assert torch.equal(_native.moe_grouped_gemm(a, w, offsets, P, order, row_div, act=act), _native.moe_grouped_gemm(near, w, offsets, P, act=act))
    for act in (("silu",), ("clamped", 2.0, 1.702)):
        assert torch.equal(_native.moe_grouped_glu(a, w, offsets, P, order, row_div, *act), _native.moe_grouped_glu(near, w, offsets, P, None, 1, *act))
