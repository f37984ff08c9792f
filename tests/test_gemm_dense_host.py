"""sp_gemm_dense_plan over the sizes that linear hands it: a tile that divides K, shares that it can serve (host code, no GPU)."""
import contextlib

import pytest
import torch


def test_plans_fit_their_products():
    from scratchpad_amd import _native
    lib = _native.load()
    steps = [256, 128, 256, 256, 256, 128, 256, 128, 64, 256, 128, 128, 64, 64] + [64] * 7
    for M in (5, 16, 17, 31, 32, 33, 64, 65, 100, 128, 192, 255, 256, 640, 1024):
        for N in (1024, 1032, 1536, 3072, 8448, 16384, 128256):
            for K in (64, 192, 512, 1024, 2048, 3584, 8192, 14336):
                for epilogue in (0, 1):
                    plan = lib.sp_gemm_dense_plan(M, N, K, epilogue)
                    tile, splits = plan & 255, plan >> 8
                    if epilogue and plan < 0:          # the plain product has shares, or no tile with its order of sums takes pairs
                        continue
                    assert plan >= 0 and tile < len(steps) and splits in (1, 2, 3, 4, 6, 8)
                    assert K % steps[tile] == 0 and K // steps[tile] >= (3 * splits if splits > 1 else 1)
                    assert splits == 1 or epilogue == 0
    for bad in ((0, 1024, 1024, 0), (64, 1024, 1000, 0), (64, 1024, 1024, 2), (64, -1, 64, 0)):
        assert lib.sp_gemm_dense_plan(*bad) == -1


@pytest.mark.parametrize("M, N, K, takes", [(4, 28672, 4096, False), (5, 28672, 4096, True), (16, 2048, 4096, False), (16, 4096, 4096, True), (17, 4096, 4096, True), (256, 4096, 4096, True), (257, 4096, 4096, False),
                                            (640, 4096, 14336, True), (1024, 4096, 14336, True), (1025, 4096, 14336, False), (512, 7168, 14336, True), (513, 7168, 14336, False), (640, 2048, 4608, False), (144, 3072, 2048, False), (192, 3072, 2048, True), (209, 3072, 2048, False), (256, 4096, 3072, True), (768, 2048, 2048, False), (769, 2048, 2048, True), (1024, 4096, 4096, True), (1025, 2048, 2048, False), (777, 2560, 2560, False), (777, 1024, 2048, False), (777, 2048, 4160, False), (64, 512, 4096, False), (64, 1024, 1000, False),
                                            (64, 2048, 4096, True), (65, 2048, 4096, False), (17, 520, 2048, True), (300, 1024, 8192, False), (95, 128256, 2048, True), (96, 128256, 2048, False),
                                            (256, 128256, 4096, True)])
def test_where_it_pays(M, N, K, takes):
    from scratchpad_amd import _native
    assert _native.dense_gemm_pays(M, N, K) is takes


@pytest.mark.parametrize("M, N, K, takes", [
    # 769 - 1024 rows: too few tiles for a long K, tiles that fill the units, fewer for a short K
    (777, 3072, 3072, False), (900, 3072, 3072, False), (777, 3584, 4096, False), (900, 3328, 3072, True), (777, 4096, 4096, True), (777, 1536, 1024, True),
    (777, 1536, 3072, False), (1024, 1408, 4096, False), (777, 3072, 2048, True), (928, 2048, 1024, True),
    # long K: past 640 rows
    (640, 4096, 8192, True), (704, 4096, 8192, False), (768, 6144, 16384, True), (1024, 6144, 16384, False), (832, 5504, 14720, False),
    # 5 - 16 rows: K in steps of 256, few rows of short K or few weight rows, up to 4096 x 4096
    (8, 8192, 1088, False), (16, 8192, 1088, False), (5, 6144, 1536, False), (9, 6144, 1536, True), (5, 5120, 2048, True), (5, 2048, 4608, False),
    (5, 1536, 6144, True), (12, 4096, 2560, False), (13, 4096, 2560, True), (9, 3584, 3584, True), (16, 3584, 2560, False), (5, 16384, 2112, True),
    # heads
    (192, 49152, 4096, True), (193, 49152, 4096, False), (160, 65536, 1024, True), (161, 65536, 1024, False), (256, 32000, 4096, True), (256, 40960, 256, True)])
def test_what_measured_slower_stays_the_librarys(M, N, K, takes):
    from scratchpad_amd import _native
    assert _native.dense_gemm_pays(M, N, K) is takes


def test_linear_asks_for_every_product_that_pays():
    """what linear looks at before the call, for steps past DENSE_MAX_ROWS: more than 768 rows, or K past 5120"""
    from scratchpad_amd import _native
    for M in (257, 400, 768, 769, 900, 1024, 1025):
        for N in (1024, 2048, 3072, 4096, 6144, 8192, 28672):
            for K in (1024, 2048, 4096, 5120, 5184, 8192, 14336, 28672):
                if _native.dense_gemm_pays(M, N, K):
                    assert M <= _native.DENSE_LONG_ROWS and (M > 768 or K > 5120)


class _OnDevice(torch.Tensor):
    """a tensor that says it is on GPU `device`, for what looks at that and launches nothing"""
    device_index = 0
    is_cuda = True

    def get_device(self):
        return self.device_index


def _own_product(monkeypatch, device=0, current=0, dtype=torch.bfloat16, within=contextlib.nullcontext):
    """whether _dense_product, called under `within`, hands x @ w.T of 64 rows to the native product"""
    from scratchpad_amd import _native
    calls = []

    class Library:
        sp_gemm_dense_plan = staticmethod(lambda *a: 256)
        sp_gemm_dense = staticmethod(lambda *a: calls.append(a) or 0)

    with monkeypatch.context() as m:
        m.setattr(_native, "load", lambda: Library)
        m.setattr(_native, "_PLAIN", (_OnDevice,))
        m.setattr(_native, "_DENSE_PLANS", {})
        m.setattr(_native, "_DENSE_ON", True)
        m.setattr(_native, "_stream", lambda: 0)
        m.setattr(torch._C, "_cuda_getDevice", lambda: current, raising=False)
        x, w = (torch.zeros(rows, 1024, dtype=dtype).as_subclass(_OnDevice) for rows in (64, 1024))
        x.device_index = w.device_index = device
        with within():
            out = _native._dense_product(x, w, 0)
    assert (out is None) == (not calls)
    return bool(calls)


def test_only_tensors_of_the_current_device(monkeypatch):
    """the launch is on the current device's stream: a product on another one is the library's, which sets the device itself"""
    assert _own_product(monkeypatch)
    assert _own_product(monkeypatch, device=1, current=1)
    assert not _own_product(monkeypatch, device=1, current=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, N, K", [(8, 6144, 2048), (64, 768, 1024), (200, 1024, 1024), (800, 2048, 1024), (260, 2048, 5184)])
def test_tensors_that_are_not_on_a_gpu_need_no_library(monkeypatch, rows, N, K, dtype):
    from scratchpad_amd import _native

    def missing():
        raise RuntimeError("not built")

    monkeypatch.setattr(_native, "load", missing)
    monkeypatch.setattr(_native, "_DENSE_PLANS", {})
    assert _native.dense_gemm_pays(rows, N, K)
    x, w = torch.ones(rows, K, dtype=dtype), torch.ones(N, K, dtype=dtype)
    assert torch.equal(_native.linear(x, w), torch.nn.functional.linear(x, w))
    assert _native.linear(x.to("meta"), w.to("meta")).shape == (rows, N)
    assert _native.dense_silu_mul(x, w) is None and _native.linear_silu_mul(x, w) is None


def test_traced_and_symbolic_sizes():
    """sizes that are no plain numbers reach neither the table of plans nor the library"""
    from torch.fx.experimental.proxy_tensor import make_fx
    from scratchpad_amd import _native
    x, w = torch.randn(64, 1024), torch.randn(256, 1024)
    want = torch.nn.functional.linear(x, w)
    before = dict(_native._DENSE_PLANS)
    assert torch.allclose(torch.jit.trace(_native.linear, (x, w))(x, w), want)
    assert torch.allclose(make_fx(_native.linear, tracing_mode="symbolic")(x, w)(x, w), want)
    assert _native._DENSE_PLANS == before


def test_a_library_of_before_the_product():
    """its entry is a stub that raises: the products are the library's"""
    from scratchpad_amd import _native

    class Older:
        sp_gemm_dense_plan = staticmethod(_native._not_built("sp_gemm_dense_plan"))

    with pytest.MonkeyPatch.context() as m:
        m.setattr(_native, "load", lambda: Older)
        m.setattr(_native, "_DENSE_PLANS", {})
        assert _native.dense_gemm_pays(64, 1024, 1024) and _native._dense_plan(64, 1024, 1024, 0) == -1


def test_compiled_graphs_hold_the_product():
    """Dynamo traces linear as one graph, whatever the library would take"""
    from scratchpad_amd import _native
    x, w = torch.randn(64, 1024), torch.randn(1024, 1024)
    compiled = torch.compile(_native.linear, backend="eager", fullgraph=True)
    assert torch.equal(compiled(x, w), torch.nn.functional.linear(x, w))


class _Counting(torch.overrides.TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_function_modes_see_the_product(monkeypatch):
    """a mode that overrides torch's functions finds the library's product; the one that only says where new tensors go hides none"""
    assert not _own_product(monkeypatch, within=_Counting)
    assert _own_product(monkeypatch, within=lambda: torch.device("cpu"))


@contextlib.contextmanager
def _autocast(dtype):
    """torch.autocast("cuda", dtype) where there is no GPU for it to ask"""
    enabled, before = torch.is_autocast_enabled("cuda"), torch.get_autocast_dtype("cuda")
    torch.set_autocast_enabled("cuda", True)
    torch.set_autocast_dtype("cuda", dtype)
    try:
        yield
    finally:
        torch.set_autocast_enabled("cuda", enabled)
        torch.set_autocast_dtype("cuda", before)


def test_autocast_to_the_other_type_is_the_librarys(monkeypatch):
    for dtype, other in ((torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)):
        assert not _own_product(monkeypatch, dtype=dtype, within=lambda: _autocast(other))
        assert _own_product(monkeypatch, dtype=dtype, within=lambda: _autocast(dtype))


def _touch(kind, mlp, seen):
    """something of a user's that calling gate_up_proj or act_fn runs"""
    note = lambda *a: seen.append(kind)                            # noqa: E731
    if kind == "forward hook":
        mlp.gate_up_proj.register_forward_hook(lambda m, a, out: note())
    elif kind == "pre-hook":
        mlp.gate_up_proj.register_forward_pre_hook(lambda m, a: note())
    elif kind == "activation's hook":
        mlp.act_fn.register_forward_hook(lambda m, a, out: note())
    elif kind == "hook of all modules":
        return torch.nn.modules.module.register_module_forward_hook(lambda m, a, out: note())
    elif kind == "its own forward":
        before = mlp.gate_up_proj.forward
        mlp.gate_up_proj.forward = lambda x: (note(), before(x))[1]
    else:                                                           # another module in its place
        class Adapter(torch.nn.Module):
            def __init__(self, inner):
                super().__init__()
                self.inner, self.weight = inner, inner.weight

            def forward(self, x):
                note()
                return self.inner(x)

        mlp.gate_up_proj = Adapter(mlp.gate_up_proj)


@pytest.mark.parametrize("kind", ["forward hook", "pre-hook", "activation's hook", "hook of all modules", "its own forward", "adapter"])
@pytest.mark.parametrize("rows", [5, 9, 64])
def test_fused_mlp_passes_by_nothing_that_its_modules_would_run(monkeypatch, kind, rows):
    from scratchpad_amd import _native, distributed
    from scratchpad_amd.llama import LlamaMLP
    if not distributed.model_parallel_is_initialized():
        distributed.initialize_model_parallel(1)
    fused = []
    one_launch = lambda x, w: fused.append(1) or x.new_zeros(x.shape[0], w.shape[0] // 2)          # noqa: E731
    monkeypatch.setattr(_native, "linear_silu_mul", lambda x, w: one_launch(x, w) if x.shape[0] <= 8 else None)
    monkeypatch.setattr(_native, "dense_silu_mul", one_launch)
    monkeypatch.setattr(_native, "silu_and_mul", lambda x: x[:, :x.shape[1] // 2])
    mlp = LlamaMLP(64, 96, "silu", torch.float32)
    for p in mlp.parameters():
        p.data.zero_()
    mlp(torch.zeros(rows, 64))
    assert fused == [1]
    seen = []
    handle = _touch(kind, mlp, seen)
    try:
        mlp(torch.zeros(rows, 64))
    finally:
        if handle is not None:
            handle.remove()
    assert seen and fused == [1]


def test_more_work_than_a_launch_holds_is_refused():
    """2^32 threads, though every operand is within reach of its 32-bit offsets (nothing is launched: no pointer is looked at)"""
    from scratchpad_amd import _native
    lib = _native.load()
    K, bf16, unsupported = 256, 2, -2
    for tile, M, N in ((2, 1 << 19, 1 << 18), (14, 1 << 22, 1 << 15), (2, 1 << 22, 1 << 14)):
        assert lib.sp_gemm_dense(16, 16, 16, None, 0, M, N, K, K, K, N, 0, tile + 256, bf16, None) == unsupported
    M, N = 1 << 22, 1 << 13                                                                       # the sum of the shares
    assert lib.sp_gemm_dense(16, 16, 16, 16, 2 * M * N, M, N, K, K, K, N, 0, 17 + 512, bf16, None) == unsupported


def test_rows_like_a_subclass_are_plain_tensors():
    """what the own products of few rows write into: a tensor, whatever x is, with the spare rows behind it"""
    from scratchpad_amd import _native
    x = torch.zeros(3, 64, dtype=torch.bfloat16)
    for like in (x, torch.nn.Parameter(x, requires_grad=False), x.as_subclass(_OnDevice)):
        out = _native._rows_like(like, 3, 8)
        assert type(out) is torch.Tensor and out.shape == (3, 8) and out.stride() == (8, 1) and out.dtype == x.dtype
        assert out.untyped_storage().nbytes() == (3 + _native.ROW_SLACK) * 8 * 2
