"""CPU tests of the host-side mirror: pools/allocator against the reference's recorded trace,
ForwardMode semantics, rope cache construction, TP shard math, graph buckets."""
import numpy as np
import pytest
import torch

from scratchpad_amd import distributed as dist_
from scratchpad_amd.forward_info import CaptureHiddenMode, ForwardMode
from scratchpad_amd.layers import get_rope
from scratchpad_amd.model_runner import ModelConfig, ServerArgs, get_batch_sizes_to_capture
from scratchpad_amd.pool import KVCache, MHATokenToKVPool, ReqToTokenPool, TokenToKVPoolAllocator
from tests import golden


def test_allocator_trace_matches_reference():
    g = golden.load("kv_pool")
    alloc = TokenToKVPoolAllocator(16, torch.float32, "cpu", None)
    assert alloc.free_slots.dtype == torch.int64 and alloc.page_size == 1
    a0 = alloc.alloc(5)
    a1 = alloc.alloc(4)
    assert alloc.available_size() == int(g["alloc_avail0"])
    alloc.free(a0[1:3])
    a2 = alloc.alloc(8)
    assert (alloc.alloc(100) is None) == bool(g["alloc_too_many_is_none"])
    state = alloc.backup_state()
    a3 = alloc.alloc(1)
    alloc.restore_state(state)
    a4 = alloc.alloc(1)
    alloc.free_group_begin()
    alloc.free(a1[:2])
    alloc.free(a2[:3])
    assert alloc.available_size() == int(g["alloc_avail_in_group"])
    alloc.free_group_end()
    for name, val in (("a0", a0), ("a1", a1), ("a2", a2), ("a3", a3), ("a4", a4)):
        assert np.array_equal(val.numpy(), g["alloc_" + name]), name
    assert np.array_equal(alloc.free_slots.numpy(), g["alloc_free_final"])
    alloc.free(torch.empty(0, dtype=torch.int64))          # no-op
    alloc.clear()
    assert np.array_equal(alloc.free_slots.numpy(), g["alloc_free_after_clear"])
    assert 0 not in alloc.free_slots.tolist(), "slot 0 is the reserved dummy slot"


def test_req_to_token_pool_trace_matches_reference():
    g = golden.load("kv_pool")
    r2t = ReqToTokenPool(5, 12, "cpu", False)
    assert r2t.req_to_token.dtype == torch.int32
    r0 = r2t.alloc(2)
    r1 = r2t.alloc(2)
    r2t.free(r0[0])
    r2 = r2t.alloc(2)
    assert (r2t.alloc(3) is None) == bool(g["r2t_none"])
    r2t.write((torch.tensor([1, 3]), torch.tensor([4, 7])), torch.tensor([11, 13], dtype=torch.int32))
    r2t.write((2, slice(0, 3)), torch.tensor([5, 6, 7], dtype=torch.int32))
    assert r0 == g["r2t_r0"].tolist() and r1 == g["r2t_r1"].tolist() and r2 == g["r2t_r2"].tolist()
    assert np.array_equal(r2t.req_to_token.numpy(), g["r2t_table"])
    assert r2t.available_size() == int(g["r2t_avail"])
    rec = ReqToTokenPool(3, 4, "cpu", True)
    rec.write((0, slice(0, 2)), torch.tensor([9, 8], dtype=torch.int32))
    records = rec.get_write_records()
    other = ReqToTokenPool(3, 4, "cpu", False)
    other.apply_write_records(records)
    assert torch.equal(other.req_to_token, rec.req_to_token) and rec.get_write_records() == []


@pytest.mark.parametrize("interleave", [True, False])
def test_kv_pool_layout_and_guards(interleave, monkeypatch):
    monkeypatch.setattr(MHATokenToKVPool, "interleave_kv", interleave)
    pool = MHATokenToKVPool(10, 1, torch.bfloat16, 2, 64, 3, "cpu")
    assert isinstance(pool, KVCache)
    k = pool.get_key_buffer(1)
    kb, vb = pool.get_kv_buffer(0)
    assert kb.data_ptr() != vb.data_ptr()
    assert k.shape == (11, 2, 64) and k.stride()[1:] == (64, 1), "[size+1, Hkv, D] token-major"
    if interleave:
        # ONE arena [layers, size+1, 2, Hkv, D]: a token's K row and V row of a layer are adjacent
        assert k.stride(0) == 256
        assert vb.data_ptr() - kb.data_ptr() == 128 * 2
        assert pool.get_key_buffer(2).data_ptr() - pool.get_key_buffer(1).data_ptr() == 11 * 256 * 2
        kb[3].fill_(1.0)
        vb[3].fill_(2.0)
        assert pool._kv_arena[0, 3].flatten().tolist() == [1.0] * 128 + [2.0] * 128
    else:
        # one arena per K/V: layer l is a view at l * (size+1) rows
        assert k.stride(0) == 128
        assert pool.get_key_buffer(2).data_ptr() - pool.get_key_buffer(1).data_ptr() == 11 * 128 * 2
    assert pool.get_kv_size_bytes() == (3 * 11 * 128 * 2,) * 2
    # the flat-data / transfer pair keeps the reference's semantics (memory/pool.py:348-372) on either layout
    idx = torch.tensor([2, 5, 9])
    for l in range(3):
        pool.k_buffer[l][idx] = torch.randn(3, 2, 64).to(torch.bfloat16)
        pool.v_buffer[l][idx] = torch.randn(3, 2, 64).to(torch.bfloat16)
    flat = pool.get_flat_data(idx)
    assert flat.shape == (2, 3, 3, 2, 64) and torch.equal(flat[0, 1], pool.get_key_buffer(1)[idx])
    other = MHATokenToKVPool(10, 1, torch.bfloat16, 2, 64, 3, "cpu")
    other.transfer(idx, flat)
    assert torch.equal(other.get_value_buffer(2)[idx], pool.get_value_buffer(2)[idx])
    other.transfer_per_layer(torch.tensor([1]), torch.stack([kb[3:4], vb[3:4]]), 1)
    assert torch.equal(other.get_key_buffer(1)[1], kb[3]) and torch.equal(other.get_value_buffer(1)[1], vb[3])
    # memory/pool.py:329-346: the transfer engines upstream address token i of buffer b at ptrs[b] + i * items[b]; walk
    # that contract with ctypes over every listed buffer and compare with the views the kernels use
    import ctypes
    ptrs, lens, items = pool.get_contiguous_buf_infos()
    rows = {}
    for b, (ptr, n, item) in enumerate(zip(ptrs, lens, items)):
        assert n == 11 * item
        for tok in (0, 3, 10):
            raw = (ctypes.c_uint16 * (item // 2)).from_address(ptr + tok * item)
            rows[b, tok] = torch.frombuffer(bytearray(raw), dtype=torch.bfloat16).clone()
    regions = sorted((p_, p_ + n) for p_, n in zip(ptrs, lens))
    assert all(a[1] <= b_[0] for a, b_ in zip(regions, regions[1:])), "listed buffers must not overlap"
    if interleave:
        assert len(ptrs) == 3 and items == [512] * 3                  # one K|V pair per token per layer
        for l in range(3):
            for tok in (0, 3, 10):
                assert torch.equal(rows[l, tok][:128], pool.get_key_buffer(l)[tok].flatten())
                assert torch.equal(rows[l, tok][128:], pool.get_value_buffer(l)[tok].flatten())
    else:
        assert len(ptrs) == 6 and items == [256] * 6                  # K buffers, then V buffers, as upstream
        for l in range(3):
            for tok in (0, 3, 10):
                assert torch.equal(rows[l, tok], pool.get_key_buffer(l)[tok].flatten())
                assert torch.equal(rows[3 + l, tok], pool.get_value_buffer(l)[tok].flatten())
    with pytest.raises(NotImplementedError):
        MHATokenToKVPool(10, 16, torch.bfloat16, 2, 64, 1, "cpu")
    with pytest.raises(RuntimeError, match="no CPU fallback"):   # the store itself is HIP-only
        from types import SimpleNamespace
        pool.set_kv_buffer(SimpleNamespace(layer_id=0), torch.tensor([1]), torch.zeros(1, 2, 64, dtype=torch.bfloat16),
                           torch.zeros(1, 2, 64, dtype=torch.bfloat16))


def test_forward_mode_semantics():
    # forward_info.py:38-66 (the reference compares against the raw ints 1..7)
    assert [int(m) for m in ForwardMode] == [1, 2, 3, 4, 5, 6, 7]
    assert ForwardMode.EXTEND.is_extend() and ForwardMode.MIXED.is_extend()
    assert not ForwardMode.DECODE.is_extend() and ForwardMode.DECODE.is_decode()
    assert ForwardMode.MIXED.is_mixed() and ForwardMode.IDLE.is_idle()
    assert ForwardMode.DECODE.is_cuda_graph() and ForwardMode.IDLE.is_cuda_graph()
    assert ForwardMode.TARGET_VERIFY.is_cuda_graph() and not ForwardMode.EXTEND.is_cuda_graph()
    assert ForwardMode.IDLE.is_decode_or_idle() and ForwardMode.DUMMY_FIRST.is_dummy_first()
    assert not CaptureHiddenMode.NULL.need_capture() and CaptureHiddenMode.LAST.is_last()


def test_rope_cache_is_the_references_bit_for_bit():
    g = golden.load("rotary")
    for i in range(int(g["num_cases"])):
        sc = golden.rope_scaling(g, i)          # None, llama3, or (round 4) linear / dynamic NTK / YaRN
        rope = get_rope(int(g[f"c{i}_head_size"]), int(g[f"c{i}_rotary_dim"]), int(g[f"c{i}_max_pos"]),
                        float(g[f"c{i}_base"]), bool(g[f"c{i}_neox"]), sc, dtype=torch.float32)
        assert np.array_equal(rope.cos_sin_cache.numpy(), g[f"c{i}_cos_sin_cache"]), f"case {i} {sc}"
    a = get_rope(64, 64, 128, 10000, True, None, torch.float32)
    assert a is get_rope(64, 64, 128, 10000, True, None, torch.float32), "cached per key"
    assert get_rope(64, 64, 128, 10000, True, None, torch.float32, partial_rotary_factor=0.5).rotary_dim == 32
    kinds = [golden.rope_scaling(g, i)["rope_type"] for i in range(int(g["num_cases"])) if golden.rope_scaling(g, i)]
    assert sorted(set(kinds)) == ["dynamic", "linear", "llama3", "yarn"]
    for unbuilt in ("deepseek_yarn", "longrope"):           # MLA / Phi-3 model families: out of scope
        with pytest.raises(ValueError):
            get_rope(64, 64, 128, 10000, True, {"rope_type": unbuilt, "factor": 2.0}, torch.float32)
    with pytest.raises(NotImplementedError):                 # per-LoRA tables (a list of linear factors)
        get_rope(64, 64, 128, 10000, True, {"rope_type": "linear", "factor": [2.0, 4.0]}, torch.float32)


def test_model_config_head_math_and_graph_buckets():
    c8, c70 = ModelConfig.llama3_8b(), ModelConfig.llama3_70b()
    assert (c8.head_dim, c8.get_num_kv_heads(1), c8.get_num_kv_heads(8), c8.get_num_kv_heads(16)) == (128, 8, 1, 1)
    assert c70.num_attention_heads // 8 == 8 and c70.get_num_kv_heads(8) == 1
    assert ModelConfig.llama32_1b().head_dim == 64
    assert get_batch_sizes_to_capture(ServerArgs(cuda_graph_max_bs=160), 4096) == \
        [1, 2, 4, 8] + list(range(16, 161, 8))          # the reference's list (cuda_graph_runner.py:100)
    assert get_batch_sizes_to_capture(ServerArgs(), 4096)[-1] == 256
    assert get_batch_sizes_to_capture(ServerArgs(cuda_graph_bs=[4, 300, 64]), 100) == [4, 64]


def test_runner_refuses_to_run_without_a_gpu():
    if torch.cuda.is_available():
        pytest.skip("GPU present")
    from scratchpad_amd.model_runner import ModelRunner
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ModelRunner(ModelConfig(64, 128, 1, 2, 1, 100))
    with pytest.raises(RuntimeError, match="unsupported device"):
        ModelRunner(ModelConfig(64, 128, 1, 2, 1, 100), device="cpu")


def test_qkv_shard_math_single_rank():
    """tp=1: the merged layout is [q | k | v] (linear.py:746-760)"""
    dist_.destroy_model_parallel()
    dist_.initialize_model_parallel(1)
    from scratchpad_amd.llama import MergedColumnParallelLinear, QKVParallelLinear, RowParallelLinear
    qkv = QKVParallelLinear(64, 16, 4, 2)
    assert (qkv.num_heads, qkv.num_kv_heads, qkv.num_kv_head_replicas) == (4, 2, 1)
    assert qkv.weight.shape == ((4 + 2 * 2) * 16, 64)
    full = torch.arange(128 * 64, dtype=torch.float32).view(128, 64)
    assert torch.equal(qkv.shard_from_full(full), full)
    assert MergedColumnParallelLinear(64, [96, 96]).weight.shape == (192, 64)
    assert RowParallelLinear(96, 64).weight.shape == (64, 96)
    dist_.destroy_model_parallel()


# ---------------------------------------------------------------- host logic added with the §8f rows
def test_sampling_params_and_batch_info_host_side():
    import torch
    from scratchpad_amd.sampler import TOP_K_ALL, SamplingBatchInfo, SamplingParams
    greedy = SamplingParams(temperature=0.0)
    assert greedy.top_k == 1 and greedy.temperature == 1.0          # sampling_params.py:66-69
    assert SamplingParams(top_k=-1).top_k == TOP_K_ALL               # whole vocabulary
    for bad in (dict(top_p=0.0), dict(top_p=1.5), dict(min_p=-0.1), dict(temperature=-1.0), dict(top_k=0)):
        with pytest.raises(ValueError):
            SamplingParams(**bad).verify()
    a = SamplingBatchInfo.from_params([greedy, SamplingParams(temperature=0.7, top_k=40, min_p=0.05)], 100, "cpu")
    b = SamplingBatchInfo.from_params([greedy], 100, "cpu")
    assert not a.is_all_greedy and a.need_min_p_sampling and b.is_all_greedy and not b.need_min_p_sampling
    assert a.temperatures.shape == (2, 1) and a.top_ks.dtype == torch.int32 and len(a) == 2
    a.merge_batch(b)
    assert len(a) == 3 and a.top_ks.tolist() == [1, 40, 1] and not a.is_all_greedy
    a.filter_batch([0, 2], torch.tensor([0, 2]))
    assert len(a) == 2 and a.top_ks.tolist() == [1, 1] and a.min_ps.tolist() == [0.0, 0.0]


def test_skinny_gemm_dispatch_rule_and_cpu_passthrough():
    import torch
    from scratchpad_amd import _native
    pays = _native.skinny_gemm_pays
    assert pays(1, 6144, 4096) and pays(1, 28672, 4096) and pays(1, 128256, 4096)       # bs 1: all but down_proj
    assert pays(16, 4096, 4096) and pays(8, 6144, 4096) and pays(8, 28672, 4096)
    assert not pays(1, 4096, 14336) and not pays(8, 4096, 14336)                          # long rows: library
    assert not pays(16, 28672, 4096) and not pays(8, 128256, 4096)
    x, w = torch.randn(3, 64), torch.randn(5, 64)
    assert torch.equal(_native.linear(x, w), torch.nn.functional.linear(x, w))           # host tensors: plain F.linear


def test_skinny_gemm_takes_the_head_of_few_rows():
    from scratchpad_amd import _native
    pays = _native.skinny_gemm_pays
    assert all(pays(m, 128256, k) for m in (1, 3, 4) for k in (2048, 4096)) and pays(8, 128256, 2048)
    assert not pays(5, 128256, 4096) and not pays(9, 128256, 2048) and not pays(3, 4096, 14336)


def test_skinny_gemm_leaves_large_heads_of_short_rows_to_the_library():
    from scratchpad_amd import _native
    pays = _native.skinny_gemm_pays
    assert not pays(8, 128256, 1024) and not pays(5, 128256, 1536) and not pays(8, 262144, 1024)
    assert pays(4, 128256, 1024) and pays(8, 128256, 512) and pays(8, 65536, 1024)


def test_delta_chunk_dispatch_rule():
    """chunks where they measured faster than the walk token by token: not for portions of 8 (18) tokens whatever the head"""
    from scratchpad_amd import _native
    least = _native.delta_chunk_tokens
    assert least(True, 128, 128, 128) == 8 and least(True, 1024, 128, 128) == 8 and least(False, 1024, 128, 128) == 8
    assert least(True, 256, 128, 128) > 17 and least(True, 64, 64, 64) > 24 and least(True, 512, 128, 64) > 40
    assert least(False, 64, 128, 128) > 20 and least(False, 512, 64, 64) > 40 and least(False, 4096, 128, 64) > 33
    assert all(8 <= least(c, W, D, Dv) <= 56 for c in (True, False) for W in (1, 64, 256, 1024, 8192) for D in (64, 128) for Dv in (16, 64, 128, 256))


def test_fp32_product_dispatch_rule():
    """the tiles for many bf16 rows where they measured faster than the library, the library where it did"""
    from scratchpad_amd import _native
    pays = _native.small_linear_tiles_pay
    assert pays(65, 2048, 32) and pays(16384, 2048, 64) and pays(8192, 2048, 128) and pays(4096, 2048, 256) and pays(256, 2048, 1024)
    assert pays(512, 4096, 64) and pays(2048, 4096, 256) and pays(1024, 8192, 64)
    assert pays(65, 4096, 64) and pays(256, 4096, 16) and pays(512, 8192, 64) and pays(65, 4096, 2048)       # a long chain, few rows
    assert pays(8192, 2048, 256) and pays(4096, 2048, 512) and pays(4096, 4096, 256) and pays(256, 2048, 2048)
    assert not pays(16384, 64, 256) and not pays(32768, 64, 64) and not pays(32768, 256, 512)                # many outputs of many rows, short and
    assert not pays(8192, 4096, 512) and not pays(777, 4096, 2048) and not pays(16384, 16384, 100)           # long


def test_fp32_products_of_far_apart_rows_leave_the_tiles():
    """a tile's loads count in 32 bits from its first row: 64 rows of the widest stride that takes tiles lie within them"""
    from scratchpad_amd import _native
    w = torch.empty(64, 2048, device="meta")
    rows = lambda stride: torch.empty_strided((65, 2048), (stride, 1), dtype=torch.bfloat16, device="meta")  # noqa: E731
    widest = max(s for s in (2048, 1 << 20, 1 << 25, (1 << 25) + 8, 34087048, 69273672) if _native._small_linear_tiles_take(rows(s), w))
    assert widest >= 1 << 20 and 63 * widest * 2 + 128 <= 1 << 32
    assert not _native._small_linear_tiles_take(rows(34087048), w) and not _native._small_linear_tiles_take(rows(69273672), w)


def test_scan_segments_keep_to_one_round_and_to_long_requests():
    """a step is cut only where its longest request is likely to be several segments, into multiples of 64 tokens whose workgroups the
    chip holds at a time"""
    from scratchpad_amd import _native
    rule = _native._scan_segment
    for tokens in (1, 64, 300, 448, 1000, 3001, 4096, 16384, 100000):
        for requests in (1, 2, 5, 8, 16, 300):
            for heads in (1, 8, 16, 64, 300):
                for slots, least in ((256, 448), (512, 800)):
                    n = rule(tokens, requests, heads, slots, least)
                    if n:
                        assert n % 64 == 0 and n >= 128 and tokens >= least and 7 * n <= 4 * tokens // requests
                        assert (tokens / n + requests / 2) * heads <= slots
    assert rule(4096, 1, 16, 256, 448) and rule(3001, 5, 16, 256, 448) and rule(4096, 1, 64, 512, 800)
    assert not rule(4096, 8, 16, 256, 448) and not rule(300, 1, 16, 256, 448) and not rule(4096, 4, 64, 512, 800)


def test_rules_of_the_recurrences_take_steps_without_requests():
    """an empty step (a batch that was filtered away) asks the same rules"""
    from scratchpad_amd import _native
    assert _native._scan_segment(0, 0, 16, 256, 448) == 0 and _native._hgrn2_segment(0, 0, 8) == 0
    assert not _native.hgrn2_chunks_pay(0, 0, 8) and not _native.delta_recurrence_chunks_pay(0, 0, 32)
    assert not _native.hgrn2_chunks_pay(0, 3, 8) and _native._scan_segment(0, 3, 16, 256, 448) == 0      # requests of no tokens


def test_rules_of_the_recurrences_know_the_longest_request(monkeypatch):
    """a forward batch's lengths are on the host: the forms for long requests are taken where one is long and not where twice the mean
    would be, and where the lengths are not known the guess stays"""
    from scratchpad_amd import _native
    from scratchpad_amd.forward_info import ForwardBatch, ForwardMode
    monkeypatch.setattr(_native, "_gpu", lambda *a: None)
    monkeypatch.setattr(_native, "token_requests", lambda starts, n: torch.zeros(n, dtype=torch.int32))
    ints = lambda v, dt=torch.int32: torch.tensor(v, dtype=dt)  # noqa: E731

    def params(lens, known=True):
        n = len(lens)
        fb = ForwardBatch(forward_mode=ForwardMode.EXTEND, batch_size=n, input_ids=ints([0] * sum(lens), torch.int64),
                          req_pool_indices=ints(list(range(n)), torch.int64), seq_lens=ints(lens, torch.int64),
                          out_cache_loc=ints([0] * sum(lens), torch.int64), seq_lens_sum=sum(lens))
        fb.extend_num_tokens, fb.extend_seq_lens, fb.extend_prefix_lens = sum(lens), ints(lens), ints([0] * n)
        fb.extend_start_loc = ints([sum(lens[:i]) for i in range(n)])
        fb.extend_seq_lens_cpu = list(lens) if known else None
        return _native.SeqParams.from_forward_batch(fb)
    assert params([3, 70, 5]).longest == 70 and params([3, 70, 5], False).longest is None
    rule = lambda r, lens, *more: r(sum(lens), len(lens), *more, longest=params(lens).longest)  # noqa: E731
    mlstm, mamba2 = (256, 448), (512, 576)
    cut = lambda parts: lambda *a, **k: _native._scan_segment(*a, **k, parts=parts)  # noqa: E731
    for lens in ([230] * 2, [300] * 4, [300] * 8):
        assert not rule(cut(2.5), lens, 8, *mlstm)
    for lens in ([500] * 3, [1000] * 3, [4000] * 3):
        assert not rule(cut(2.75), lens, 64, *mamba2)
    for lens in ([40] * 8, [60] * 4, [40] * 32, [16] * 64):
        assert not rule(_native.hgrn2_chunks_pay, lens, 8)
    assert not rule(_native.delta_recurrence_chunks_pay, [40] * 16, 32) and not rule(_native.delta_recurrence_chunks_pay, [100] * 32, 32)
    uneven = [2000] + [3] * 60                     # one prompt among the portions of a running batch
    assert rule(_native.hgrn2_chunks_pay, uneven, 8) and rule(_native._hgrn2_segment, uneven, 8)
    assert rule(_native.delta_recurrence_chunks_pay, uneven, 32) and rule(cut(2.5), [4000] + [10] * 7, 16, *mlstm)


def test_mlstm_scan_takes_no_gate_rows_that_overlap(monkeypatch):
    """gates whose rows lie closer than their width (an expanded row, a sliding view) are refused before anything is launched: the
    kernel reads [token, head] at rows at least `heads` apart.  Views of one product and strides that differ pass."""
    import types

    import torch
    from scratchpad_amd import _native

    class DeviceTensor(torch.Tensor):
        is_cuda = True

    calls = []
    lib = types.SimpleNamespace(sp_mlstm_scan_tokens=lambda *a: calls.append(a) or 0)
    monkeypatch.setattr(_native, "load", lambda: lib)
    monkeypatch.setattr(_native, "_stream", lambda: 0)
    T, H, D = 6, 4, 16
    dev = lambda *shape: torch.randn(*shape).as_subclass(DeviceTensor)  # noqa: E731
    q, k, v, g = (dev(T, H * D) for _ in range(4))
    nw, S, n, m = dev(H * D), dev(3, H, D, D), dev(3, H, D), dev(3, H)
    seq = types.SimpleNamespace(num_tokens=T, batch_size=1, extend_seq_lens=object(), args=())
    scan = lambda i, f: _native.mlstm_scan(q, k, v, g, i, f, nw, S, n, m, seq, H, D, D, 15.0, 1e-5)  # noqa: E731
    both, row = dev(T, 2 * H), dev(1, H)
    for i, f, stride in ((dev(T, H), dev(T, H), H), (both[:, :H], both[:, H:], 2 * H), (both[:, :H], dev(T, H), H)):
        scan(i, f)
        assert calls.pop()[12] == stride
    near = dev(T + H).as_strided((T, H), (1, 1))
    for i, f in ((row.expand(T, H), row.expand(T, H)), (row.expand(T, H), dev(T, H)), (near, near), (dev(T, H), near)):
        with pytest.raises(RuntimeError):
            scan(i, f)
    assert not calls


def test_vision_attention_plan_partition(monkeypatch):
    import torch
    from scratchpad_amd import vision
    from scratchpad_amd.mllama_vision import padding_positions
    monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: object())
    P, Pp = 1025, 1032
    pad = padding_positions(torch.tensor([[1, 1, 1, 1], [1, 0, 0, 0]]), P, Pp)
    assert pad.shape == (2, 4 * Pp) and int(pad[0].sum()) == 4 * 7 and int(pad[1].sum()) == 3 * Pp + 7
    plan = vision.VisionAttnPlan(2, 4 * Pp, "cpu", pad_rows=pad)
    assert plan.main.seq_lens == [4 * Pp] * 2 and plan.main_rows is None                  # natural order
    assert plan.side.seq_lens == [28, 3 * Pp + 7] and plan.side.key_lens == [4 * P, P]
    assert plan.side.key_index.shape == (2, 4 * P) and plan.side.key_index[1, P - 1] == 4 * Pp + P - 1
    assert torch.equal(plan.side_rows[:7], torch.arange(P, Pp))
    rag = vision.VisionAttnPlan(1, 10, "cpu", cu_seqlens=[0, 3, 3, 10])
    assert rag.main.seq_lens == [3, 0, 7] and rag.side is None and rag.main.start.tolist() == [0, 3, 3]
    monkeypatch.setattr(vision.VisionAttnPlan, "MOVE_SPILL_ROWS", True)
    moved = vision.VisionAttnPlan(1, 4 * Pp, "cpu", pad_rows=pad[:1])
    assert moved.main.seq_lens == [4096] and moved.side.seq_lens == [28, 4] and moved.side.key_lens == [4 * P, 4 * Pp]
    both = torch.cat([moved.main_rows, moved.side_rows]).sort().values
    assert torch.equal(both, torch.arange(4 * Pp)), "every position is computed exactly once"


def test_ring_allocators_match_a_list_model_across_wraps():
    """Both free lists are rings (pool.py): a long random alloc / free / free-group / backup-restore
    sequence, which wraps the rings many times, must hand out exactly what the reference's
    slice-the-head / append-at-the-tail lists would."""
    import random
    rnd = random.Random(7)
    size = 37
    alloc = TokenToKVPoolAllocator(size, torch.float32, "cpu", None)
    model = list(range(1, size + 1))
    held = []
    for step in range(3000):
        op = rnd.random()
        if op < 0.45:
            n = rnd.randint(0, 9)
            got = alloc.alloc(n)
            if n > len(model):
                assert got is None
            else:
                assert got.tolist() == model[:n], step
                model = model[n:]
                held.extend(got.tolist())
        elif op < 0.85 and held:
            rnd.shuffle(held)
            k = rnd.randint(1, min(len(held), 11))
            back, held = held[:k], held[k:]
            if rnd.random() < 0.3:
                alloc.free_group_begin()
                assert not alloc.is_not_in_free_group
                mid = rnd.randint(0, k)
                alloc.free(torch.tensor(back[:mid], dtype=torch.int64))
                alloc.free(torch.tensor(back[mid:], dtype=torch.int64))
                assert alloc.available_size() == len(model), "a group's frees land at free_group_end"
                alloc.free_group_end()
            else:
                alloc.free(torch.tensor(back, dtype=torch.int64))
            model = model + back
        elif op < 0.9:
            state = alloc.backup_state()
            n = min(len(model), rnd.randint(0, 5))
            assert alloc.alloc(n).tolist() == model[:n]
            alloc.restore_state(state)              # the allocation is undone
        assert alloc.available_size() == len(model)
    assert alloc.free_slots.tolist() == model and 0 not in model
    with pytest.raises(RuntimeError, match="overflow"):
        alloc.free(torch.arange(1, size + 2))

    rows = ReqToTokenPool(9, 4, "cpu")
    rmodel = list(range(9))
    rheld = []
    for step in range(2000):
        if rnd.random() < 0.5:
            n = rnd.randint(0, 4)
            got = rows.alloc(n)
            if n > len(rmodel):
                assert got is None
            else:
                assert got == rmodel[:n] and all(isinstance(x, int) for x in got)
                rmodel = rmodel[n:]
                rheld.extend(got)
        elif rheld:
            rnd.shuffle(rheld)
            if rnd.random() < 0.5:
                x = rheld.pop()
                rows.free(x)
                rmodel.append(x)
            else:
                k = rnd.randint(1, len(rheld))
                back, rheld = rheld[:k], rheld[k:]
                rows.free(back)
                rmodel.extend(back)
        assert rows.available_size() == len(rmodel) and rows.free_slots == rmodel


def test_mixed_batch_merges_sampling_info_like_the_reference():
    """mix_with_running goes through merge_batch (schedule_batch.py:1073-1101, 1361-1397): the running
    decodes' sampling parameters, pending output ids and request list are merged in request order - a
    running request that samples with temperature must not silently become greedy in a MIXED batch."""
    from scratchpad_amd.sampler import SamplingBatchInfo, SamplingParams
    from scratchpad_amd.schedule_batch import Req, ScheduleBatch

    def batches(prefill_params, running_params):
        r2t = ReqToTokenPool(8, 16, "cpu")
        alloc = TokenToKVPoolAllocator(32, torch.float32, "cpu", None)
        new = ScheduleBatch([Req("n0", "", [1, 2, 3, 4], prefill_params)], r2t, alloc, device="cpu")
        new.forward_mode = ForwardMode.EXTEND
        new.input_ids = torch.tensor([1, 2, 3, 4])
        new.out_cache_loc = torch.tensor([10, 11, 12, 13])
        new.req_pool_indices = torch.tensor([0])
        new.seq_lens = torch.tensor([4])
        new.seq_lens_sum, new.extend_num_tokens = 4, 4
        new.prefix_lens, new.extend_lens = [0], [4]
        run = ScheduleBatch([Req("r0", "", [5, 6], running_params[0], output_ids=[7]),
                             Req("r1", "", [8], running_params[1], output_ids=[9, 9])], r2t, alloc, device="cpu")
        run.forward_mode = ForwardMode.DECODE
        run.input_ids = torch.tensor([7, 9])
        run.out_cache_loc = torch.tensor([20, 21])
        run.req_pool_indices = torch.tensor([1, 2])
        run.seq_lens = torch.tensor([3, 3])
        run.seq_lens_sum = 6
        for b in (new, run):
            if any(getattr(r, "sampling_params", None) is not None for r in b.reqs):
                b.sampling_info = SamplingBatchInfo.from_schedule_batch(b, 100)
        return new, run

    hot = SamplingParams(temperature=0.7, top_k=40, top_p=0.9)
    # prefill greedy (no info at all), running requests sample: the merged info has 3 rows in request order
    new, run = batches(None, (hot, None))
    assert new.sampling_info is None and run.sampling_info is not None
    new.mix_with_running(run)
    assert new.forward_mode == ForwardMode.MIXED and [r.rid for r in new.reqs] == ["n0", "r0", "r1"]
    assert new.input_ids.tolist() == [1, 2, 3, 4, 7, 9] and new.out_cache_loc.tolist() == [10, 11, 12, 13, 20, 21]
    assert new.extend_lens == [4, 1, 1] and new.prefix_lens == [0, 2, 2] and new.extend_num_tokens == 6
    assert new.seq_lens.tolist() == [4, 3, 3] and new.seq_lens_sum == 10
    info = new.sampling_info
    assert len(info) == 3 and not info.is_all_greedy
    assert info.top_ks.tolist() == [1, 40, 1] and info.temperatures.view(-1).tolist() == pytest.approx([1.0, 0.7, 1.0])
    assert new.get_model_worker_batch().sampling_info is info
    # the other way round, and the overlap scheduler's prefix_lens (output_ids lags one step)
    new, run = batches(hot, (None, None))
    new.mix_with_running(run, enable_overlap=True)
    assert new.sampling_info.top_ks.tolist() == [40, 1, 1] and new.prefix_lens == [0, 3, 3]
    # nobody samples: the batch stays "all greedy" without materialising anything
    new, run = batches(None, (None, None))
    new.mix_with_running(run)
    assert new.sampling_info is None and len(new.reqs) == 3
    # the mixed-in running requests are extend rows of length 1 (schedule_batch.py:1077-1079), their
    # logprob bookkeeping and flags are carried (1361-1397), and pending output ids must line up or fail loudly
    new, run = batches(None, (None, None))
    run.return_logprob, run.top_logprobs_nums, run.token_ids_logprobs = True, [2, 0], [None, [3, 4]]
    run.has_grammar = True
    new.extend_logprob_start_lens = [0]
    new.mix_with_running(run)
    assert [r.extend_input_len for r in new.reqs] == [4, 1, 1]
    assert new.extend_logprob_start_lens == [0, 0, 0]
    # one id per KEPT position - the prefill row's 4 (zeros: it asked for none) + one zero per running row
    # (its next token is not known yet) - so LogitsProcessor's logprobs[arange, ids] lines up (the reference leaves
    # the list short, schedule_batch.py:1073-1101, and its scheduler never builds this batch, scheduler.py:944-949)
    assert new.extend_input_logprob_token_ids.tolist() == [0] * 6
    assert new.return_logprob and new.top_logprobs_nums == [0, 2, 0] and new.token_ids_logprobs == [None, None, [3, 4]]
    assert new.has_grammar and not new.has_stream
    new.reqs[1].init_next_round_input()                 # the pin does not outlive the round
    assert new.reqs[1].extend_input_len == 3
    new, run = batches(None, (None, None))
    new.output_ids = torch.tensor([42])
    run.output_ids = torch.tensor([7, 9])
    new.mix_with_running(run)
    assert new.output_ids.tolist() == [42, 7, 9]
    new, run = batches(None, (None, None))
    new.output_ids = torch.tensor([42])                 # one side without output ids: rows would not line up
    with pytest.raises(RuntimeError, match="output_ids"):
        new.mix_with_running(run)


def test_spare_row_views_and_library_row_table():
    """_native.extend_rows re-views an activation over more rows of its own storage only when the storage
    really extends that far; library_rows never shrinks a product and is the identity off its table."""
    import torch
    from scratchpad_amd import _native
    x = _native.empty_rows(5, 8, torch.float32, "cpu")
    assert x.shape == (5, 8) and x.is_contiguous()
    v = _native.extend_rows(x, 5 + _native.ROW_SLACK)
    assert v is not None and v.shape == (5 + _native.ROW_SLACK, 8) and v.data_ptr() == x.data_ptr()
    assert _native.extend_rows(x, 6 + _native.ROW_SLACK) is None
    assert _native.extend_rows(torch.zeros(5, 8), 6) is None
    part = torch.zeros(10, 16)[2:6, :8]                   # row-strided view in the middle of a buffer
    assert _native.extend_rows(part, 8).shape == (8, 8) and _native.extend_rows(part, 9) is None
    assert _native.extend_rows(x, 3) is x
    for (N, K), table in _native._LIBRARY_ROWS_TABLE.items():
        for M, Mp in table.items():
            assert M < Mp <= M + _native.ROW_SLACK
            if _native._LIBROWS_MODE == "table" and _native.library_versions_match():
                assert _native.library_rows(M, N, K) == Mp
    assert _native.library_rows(255, 6144, 4096) == 255 and _native.library_rows(256, 1234, 4096) == 256


def test_library_row_table_is_gated_on_the_build_it_was_measured_on(monkeypatch):
    """The (shape, M) -> M' table is a measurement of one hipBLASLt build: on another torch / HIP version, with
    SP_LIBRARY_ROWS=0, and under SP_LIBRARY_ROWS=auto before the calibration has run, nothing is substituted."""
    import importlib
    import torch
    from scratchpad_amd import _native
    try:
        monkeypatch.setenv("SP_LIBRARY_ROWS", "table")
        monkeypatch.setattr(torch, "__version__", "2.11.0+rocm7.1")
        importlib.reload(_native)
        assert not _native.library_versions_match() and _native._LIBRARY_ROWS == {}
        assert _native.library_rows(256, 6144, 4096) == 256
        rep = _native.library_rows_report()
        assert rep["versions_match"] is False and rep["substituted"] == {}
        monkeypatch.undo()
        for mode in ("0", "auto"):
            monkeypatch.setenv("SP_LIBRARY_ROWS", mode)
            importlib.reload(_native)
            assert _native._LIBROWS_MODE == mode and _native.library_rows(256, 6144, 4096) == 256
        monkeypatch.undo()
    finally:
        monkeypatch.undo()
        importlib.reload(_native)
    if _native.library_versions_match():
        assert _native.library_rows(256, 6144, 4096) == 264


def test_decode_split_size_policy_and_where_items_are_planned():
    """HipAttnBackend host logic only.  (a) _plan_chunk: about one (request, split) item per CU between MIN_CHUNK and
    MAX_CHUNK, from the host's bound on sum(seq_lens) alone (the advisory longest-request hint left in round 6).
    (b) which plans carry items at all: only where a launch of the model can read them - a shape the range kernel refuses
    (decode_ranges 0), a layer with a logit soft-cap, or a step whose line does not fit the range section."""
    from scratchpad_amd.attention import HipAttnBackend
    b = HipAttnBackend.__new__(HipAttnBackend)
    b.num_kv_head, b.head_dim = 8, 128
    dt = torch.bfloat16
    assert (b.MIN_CHUNK, b.MAX_CHUNK, b.TARGET_ITEMS) == (64, 768, 256)
    assert b._plan_chunk(553000, dt) == 768                      # the headline batch
    assert b._plan_chunk(1064 * 64, dt) == 512 and b._plan_chunk(40 * 8, dt) == 64 and b._plan_chunk(10 ** 9, dt) == 768
    b.num_kv_head = 1                                            # 70B / TP 8 rank: one workgroup per item
    assert b._plan_chunk(288000, dt) == 768
    # (b) the graph launch covers no items at all where nothing reads them
    b.max_context_len, b.decode_ranges = 8192, 256
    b.plan_items = False
    assert b._graph_slots(256) == 0 and b._ranges_for(256, 8192) == 256
    b.plan_items = True
    assert b._graph_slots(256) == max(b.GRAPH_SLOTS_FLOOR, b.GRAPH_SLOTS_PER_REQ * 256) + 256
    b.plan_items, b.decode_ranges = False, 0                     # the range kernel refuses the shape: items after all
    assert b._graph_slots(16) == b.GRAPH_SLOTS_FLOOR + 16
    b.decode_ranges, b.max_context_len = 256, 2 ** 24            # bs x (context + 16) >= 2^31: the line does not fit
    assert b._ranges_for(256, 2 ** 24) == 0 and b._graph_slots(256) > 0


def test_small_steps_pass_by_no_backend_of_its_own():
    """a small step runs neither the backend's decode methods nor, over a byte pool, the pool's store: where one of them is another's, there is none"""
    from scratchpad_amd.attention import HipAttnBackend, _plain_store
    from scratchpad_amd.pool import MHATokenToKVPool

    def few(cls, **own):
        b = cls.__new__(cls)
        b.head_dim, b.kv_dtype, b.small_steps, b.plan_items = 64, torch.bfloat16, True, False
        b.__dict__.update(own)
        return b._few_keys(1, 300)
    assert few(HipAttnBackend) and few(type("Same", (HipAttnBackend,), {"forward_extend": lambda *a, **k: None}))
    for name in ("forward", "forward_decode", "rotary_and_store", "init_forward_metadata", "init_forward_metadata_replay_cuda_graph"):
        assert not few(type("Own", (HipAttnBackend,), {name: lambda *a, **k: None})), name
        assert not few(HipAttnBackend, **{name: lambda *a, **k: None}), name
    pool = MHATokenToKVPool.__new__(MHATokenToKVPool)
    own = type("Own", (MHATokenToKVPool,), {"set_kv_buffer": lambda *a: None})
    assert _plain_store(pool) and not _plain_store(own.__new__(own))
    pool.set_kv_buffer = lambda *a: None
    assert not _plain_store(pool)


def test_plan_registry_trusts_only_live_plan_buffers():
    """_native remembers what each decode plan buffer was built with (data_ptr -> (bs, max_slots, ranges)) so that a launch
    given other values raises on the host (ABI 9).  A view of the buffer is the same plan; an entry whose tensor has died is
    dropped - the allocator may have handed the address to a buffer that was never built through decode_plan()."""
    import weakref
    from scratchpad_amd import _native
    t = torch.zeros(16, dtype=torch.int32)
    key = t.data_ptr()
    _native._BUILT_PLANS[key] = (weakref.ref(t), (4, 0, 256))
    assert _native._built_with(t) == (4, 0, 256) and _native._built_with(t[:8]) == (4, 0, 256)

    class SameAddress:                      # whatever the allocator puts at that address next
        def data_ptr(self):
            return key
    del t
    assert _native._built_with(SameAddress()) is None and key not in _native._BUILT_PLANS


def test_forward_batch_refuses_what_nothing_behind_it_reads():
    """ScheduleBatch.get_model_worker_batch forwards return_hidden_states (as CaptureHiddenMode.FULL) and
    input_embeds like the reference; nothing behind ForwardBatch.init_new reads either, so it raises instead of serving such
    a request as an ordinary one (the DP-attention refusal beside them was already there)."""
    from types import SimpleNamespace
    from scratchpad_amd.forward_info import CaptureHiddenMode, ForwardBatch, ForwardMode, ModelWorkerBatch
    runner = SimpleNamespace(device="cpu", req_to_token_pool=None, token_to_kv_pool=None, attn_backend=None)

    def batch(**kw):
        return ModelWorkerBatch(bid=0, forward_mode=ForwardMode.DECODE, input_ids=torch.zeros(2, dtype=torch.int64),
                                req_pool_indices=torch.zeros(2, dtype=torch.int64), seq_lens=torch.ones(2, dtype=torch.int64),
                                out_cache_loc=torch.zeros(2, dtype=torch.int64), seq_lens_sum=2, **kw)
    with pytest.raises(NotImplementedError, match="hidden states"):
        ForwardBatch.init_new(batch(capture_hidden_mode=CaptureHiddenMode.FULL), runner)
    with pytest.raises(NotImplementedError, match="input_embeds"):
        ForwardBatch.init_new(batch(input_embeds=torch.zeros(2, 8)), runner)
    with pytest.raises(NotImplementedError, match="DP attention"):
        ForwardBatch.init_new(batch(global_num_tokens=[2]), runner)


def test_token_requests_takes_first_rows_with_a_stride(monkeypatch):
    """the requests' first rows may be a column of a table of step lengths: the kernel, which reads them one after the other, is handed a
    copy"""
    import ctypes
    import types

    import torch
    from scratchpad_amd import _native

    class DeviceTensor(torch.Tensor):
        is_cuda = True

    seen = []
    lib = types.SimpleNamespace(sp_token_requests=lambda out, start, batch, tokens, stream: seen.append(
        list((ctypes.c_int32 * batch).from_address(start))) or 0)
    monkeypatch.setattr(_native, "load", lambda: lib)
    monkeypatch.setattr(_native, "_stream", lambda: 0)
    table = torch.tensor([[0, 3], [3, 2], [5, 4]], dtype=torch.int32).as_subclass(DeviceTensor)
    for start in (table[:, 0], table[:, 0].contiguous()):
        assert _native.token_requests(start, 9).shape == (9,)
    assert seen == [[0, 3, 5], [0, 3, 5]]


def test_no_garbage_is_collected_inside_a_graph_capture(monkeypatch):
    """a dropped runner's graphs (runner and graph runner hold each other) are the collector's; destroying one waits for the device, which
    is an error inside a capture and ends the process there"""
    import gc
    import types

    import torch
    from scratchpad_amd import _native
    from scratchpad_amd.model_runner import HipGraphRunner

    capturing, destroyed = [], []

    class Graph:
        def pool(self):
            return None

        def __del__(self):
            destroyed.append(bool(capturing))

    class Capture:
        def __init__(self, graph, **kwargs):
            pass

        def __enter__(self):
            capturing.append(1)

        def __exit__(self, *args):
            capturing.pop()

    class Stream:
        def wait_stream(self, other):
            pass

    class Entered:
        def __init__(self, stream):
            pass
        __enter__ = __exit__ = lambda self, *args: None

    for name, value in (("CUDAGraph", Graph), ("graph", Capture), ("Stream", Stream), ("current_stream", Stream), ("stream", Entered),
                        ("synchronize", lambda: None)):
        monkeypatch.setattr(torch.cuda, name, value)

    def forward(ids, positions, fb):
        if capturing:                       # as many containers as a collection of the youngest generation waits for, and more
            [[i] for i in range(4 * gc.get_threshold()[0])]
            assert not gc.isenabled()

    runner = types.SimpleNamespace(
        model=types.SimpleNamespace(forward=forward), req_to_token_pool=None, token_to_kv_pool=None,
        attn_backend=types.SimpleNamespace(init_forward_metadata_capture_cuda_graph=lambda *a: None))
    new = HipGraphRunner.__new__(HipGraphRunner)
    new.model_runner, new.is_encoder_decoder, new.seq_len_fill_value, new.pool, new.stream = runner, False, 1, None, None
    new.input_ids = new.req_pool_indices = new.seq_lens = new.out_cache_loc = new.positions = torch.zeros(2, dtype=torch.int64)
    enabled = gc.isenabled()
    gc.enable()
    try:
        gc.collect()
        old = types.SimpleNamespace(graph=Graph())
        old.itself = old
        del old
        new.capture_one_batch_size(2)
        assert gc.isenabled() and True not in destroyed
        with _native.capture_graph(None):
            with _native.capture_graph(None):
                pass
            assert not gc.isenabled()
        with pytest.raises(KeyError):
            with _native.capture_graph(None):
                raise KeyError
        assert gc.isenabled()
        gc.disable()
        with _native.capture_graph(None):
            pass
        assert not gc.isenabled()
    finally:
        (gc.enable if enabled else gc.disable)()
