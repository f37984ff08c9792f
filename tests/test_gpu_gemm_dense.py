"""sp_gemm_dense at the edges of its tiles: rows and columns that leave a remainder, the shortest K a share can have, columns that are
no multiple of a store, strided operands - against an fp32 product of the same 16-bit values: one rounding of the output type plus
the noise of fp32 sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
# rows, columns and k-step of a tile, in the order of its number
TILES = [(16, 64, 256), (16, 128, 128), (32, 16, 256), (32, 32, 256), (32, 64, 256), (32, 128, 128), (48, 32, 256), (64, 32, 128),
         (64, 64, 64), (64, 64, 256), (64, 128, 128), (96, 64, 128), (96, 128, 64), (128, 96, 64),
         (128, 64, 64), (128, 128, 64), (192, 128, 64), (256, 128, 64), (256, 96, 64), (160, 256, 64), (192, 192, 64)]


def check(got, x, w, dtype):
    ref = x.float().cpu() @ w.float().cpu().T
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (got.float().cpu() - ref).abs()
    assert bool((err <= eps * ref.abs() + 1e-4 * ref.abs().max()).all()), float(err.max())


def dense(x, w, plan, epilogue=0, out=None):
    from scratchpad_amd import _native
    M, K = x.shape
    N = w.shape[0] // 2 if epilogue else w.shape[0]
    out = torch.full((M, N), float("nan"), dtype=x.dtype, device="cuda") if out is None else out
    splits = plan >> 8
    sums = torch.empty(splits * M * N, device="cuda") if splits > 1 else None
    rc = _native.load().sp_gemm_dense(out.data_ptr(), x.data_ptr(), w.data_ptr(), _native._ptr(sums), 0 if sums is None else sums.numel(), M, N, K,
                                      x.stride(0), w.stride(0), out.stride(0), epilogue, plan, _native._dt(x), _native._stream())
    return rc, out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_tiles_at_their_edges(tile, dtype):
    bm, bn, bk = TILES[tile]
    g = torch.Generator().manual_seed(tile)
    for M, N, steps, splits in [(1, 1, 1, 1), (bm - 1, bn + 1, 2, 2), (bm, bn, 3, 1), (bm + 1, 2 * bn - 2, 5, 4), (2 * bm + 17, 3 * bn - 4, 17, 8),
                                (17, 4 * bn, 24, 1), (5 * bm + 3, 2 * bn + 4, 7, 3), (4 * bm, bn - 1, 20, 6)]:
        K = bk * steps
        x = torch.randn(M, K, generator=g).to(dtype).cuda()
        w = (torch.randn(N, K, generator=g) * 0.05).to(dtype).cuda()
        rc, got = dense(x, w, tile + 256 * splits)
        assert rc == 0
        check(got, x, w, dtype)
        assert torch.equal(got, dense(x, w, tile + 256 * splits)[1]), "fixed order of the sums"
    # views: x inside wider rows, w every other row, results into wider rows whose other columns stay
    wide = torch.randn(bm + 3, bk * 2 + 64, generator=g).to(dtype).cuda()
    w2 = (torch.randn(2 * (bn + 8), bk * 2, generator=g) * 0.05).to(dtype).cuda()
    x, w = wide[:, 64:], w2[::2]
    room = torch.full((bm + 3, bn + 13), -7.0, dtype=dtype, device="cuda")
    rc, got = dense(x, w, tile + 256, out=room[:, 1:bn + 9])
    assert rc == 0
    check(got, x, w, dtype)
    assert bool((room[:, 0] == -7).all()) and bool((room[:, bn + 9:] == -7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_epilogue_is_the_product_then_the_activation(dtype):
    """the bits of the same tile's product followed by sp_silu_and_mul"""
    from scratchpad_amd import _native
    g = torch.Generator().manual_seed(3)
    for tile, (bm, bn, bk) in enumerate(TILES):
        x = torch.randn(bm + 5, bk * 3, generator=g).to(dtype).cuda()
        w = (torch.randn(2 * (bn + bn // 2 + 3), bk * 3, generator=g) * 0.1).to(dtype).cuda()
        rc, got = dense(x, w, tile + 256, 1)
        assert rc == 0 and torch.equal(got, _native.silu_and_mul(dense(x, w, tile + 256)[1])), TILES[tile]


def test_linear_takes_it_and_leaves_the_rest():
    from scratchpad_amd import _native
    g = torch.Generator().manual_seed(5)
    for M, N, K in [(5, 6144, 2048), (16, 4096, 2560), (17, 1024, 1024), (61, 3072, 2048), (100, 2048, 8192), (256, 4096, 1024), (500, 2048, 6144), (777, 2048, 8192), (1001, 2048, 1024)]:
        assert _native.dense_gemm_pays(M, N, K)
        x = torch.randn(M, K, generator=g).bfloat16().cuda()
        w = (torch.randn(N, K, generator=g) * 0.05).bfloat16().cuda()
        got = _native.linear(x, w)
        assert torch.equal(got, dense(x, w, _native._dense_plan(M, N, K, 0))[1])
        check(got, x, w, torch.bfloat16)
        act = _native.dense_silu_mul(x, w)
        assert (act is None) == (_native._dense_plan(M, N, K, 1) < 0)
        assert act is None or torch.equal(act, _native.silu_and_mul(got)), (M, N, K)
    odd = torch.randn(61 * 1024 + 1, generator=g).bfloat16().cuda()[1:].view(61, 1024)       # not 16-byte aligned: the library
    w = (torch.randn(1024, 1024, generator=g) * 0.05).bfloat16().cuda()
    assert torch.equal(_native.linear(odd, w), torch.nn.functional.linear(odd, w))
    leaf = torch.randn(61, 1024, generator=g).bfloat16().cuda().requires_grad_()              # autograd sees the library's product
    _native.linear(leaf, w).sum().backward()
    assert leaf.grad is not None
    x = torch.randn(3, 61, 1024, generator=g).bfloat16().cuda()
    assert torch.func.vmap(lambda t: _native.linear(t, w))(x).shape == (3, 61, 1024)
    assert _native.linear(x, w).shape == (3, 61, 1024)
    rc, _ = dense(x[0], w, 0 + 256 * 5)
    assert rc == -1
    rc, _ = dense(x[0][:, :192], w[:, :192], 0 + 256)                                         # K is no multiple of the tile's step
    assert rc == -2


def test_replays_of_a_captured_product_are_the_eager_one():
    """with a sum over shares of K, replayed between eager work on the same inputs' buffer"""
    from scratchpad_amd import _native
    g = torch.Generator().manual_seed(6)
    x = torch.randn(40, 8192, generator=g).bfloat16().cuda()
    w = (torch.randn(2048, 8192, generator=g) * 0.05).bfloat16().cuda()
    assert _native._dense_plan(40, 2048, 8192, 0) >> 8 > 1
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        _native.linear(x, w)
    st.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=st):
        out = _native.linear(x, w)
    for i in range(4):
        x.copy_(torch.randn(40, 8192, generator=g).bfloat16())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, _native.linear(x, w)), i


def test_compiled_graphs_hold_the_product():
    """Dynamo traces linear of tensors on the GPU as one graph: no call into the library that it cannot see"""
    from scratchpad_amd import _native
    x, w = torch.randn(64, 1024, device="cuda").bfloat16(), torch.randn(1024, 1024, device="cuda").bfloat16()
    assert _native.dense_gemm_pays(64, 1024, 1024)
    compiled = torch.compile(_native.linear, backend="eager", fullgraph=True)
    assert torch.equal(compiled(x, w), torch.nn.functional.linear(x, w))


def test_function_modes_find_the_librarys_product():
    from scratchpad_amd import _native
    x, w = torch.randn(64, 1024, device="cuda").bfloat16(), torch.randn(1024, 1024, device="cuda").bfloat16()
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Mode():
        _native.linear(x, w)
    assert torch.nn.functional.linear in seen


def test_autocast_to_the_other_type_is_the_librarys():
    from scratchpad_amd import _native
    x, w = torch.randn(64, 1024, device="cuda").bfloat16(), torch.randn(1024, 1024, device="cuda").bfloat16()
    with torch.autocast("cuda", torch.float16):
        assert _native.linear(x, w).dtype == torch.float16


@pytest.mark.parametrize("N, K", [(4096, 6144), (6144, 8192), (18944, 14336), (6144, 2048), (4096, 4096), (28672, 4096), (2048, 1024)])
def test_silu_of_a_projection_has_the_bits_of_two_steps(N, K):
    """at the rows of small decode steps: of linear's product where sp_gemm_dense has the activation in its epilogue, else of sp_gemm_skinny's - also
    where linear takes neither (K that sp_gemm_dense shares out, K past 8192 at 1 - 4 rows)"""
    from scratchpad_amd import _native
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.randn(N, K, generator=g, device="cuda").mul_(0.05).bfloat16()
    for M in (1, 2, 4, 5, 7, 8):
        x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
        if _native._dense_plan(M, N, K, 1) >= 0:
            plain = _native.linear(x, w)
        else:
            plain = torch.empty(M, N, dtype=x.dtype, device="cuda")
            _native._check(_native.load().sp_gemm_skinny(plain.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K, K, K, N, 0, _native._dt(x),
                                                         _native._stream()), "sp_gemm_skinny")
        assert torch.equal(_native.linear_silu_mul(x, w), _native.silu_and_mul(plain)), M
