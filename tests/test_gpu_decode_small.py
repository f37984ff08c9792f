"""A layer's rotation, store and attention of a small decode step in one launch (sp_decode_small) against the oracle's three steps, and the
model's steps that take it."""
import pytest
import torch

from oracle import ops
from tests import smoke_impl
from tests.helpers import assert_attn_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bytes_pool", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 64), (6, 6, 128), (8, 1, 128), (3, 1, 64)])
# one key; the edges of a tile of 16, of the waves' first tiles together, of a pass (512 keys at 64, 256 at 128) and of two
@pytest.mark.parametrize("lens", [[1], [16, 17, 128, 129], [255, 256, 257, 2], [511, 512, 513, 1030]])
def test_one_launch_against_the_steps(dtype, bytes_pool, Hq, Hkv, D, lens):
    from scratchpad_amd import _native
    g = torch.Generator().manual_seed(sum(lens) + D + Hq)
    bs, total = len(lens), sum(lens) + 5
    perm = torch.randperm(total, generator=g) + 1
    table = torch.zeros(bs + 2, max(lens) + 3, dtype=torch.int32)
    rows, loc, at = torch.randperm(bs + 2, generator=g)[:bs], [], 0
    for r, n in zip(rows, lens):
        table[r, :n] = perm[at:at + n].int()
        loc.append(int(perm[at + n - 1]))
        at += n
    loc = torch.tensor(loc)
    pool_type = torch.float8_e5m2 if bytes_pool else dtype
    kb, vb = (torch.randn(total + 1, Hkv, D, generator=g).to(pool_type) for _ in range(2))
    for b in (kb, vb):                          # what the new slots hold is as old as their last use
        b.view(torch.uint8)[loc] = 0x7f
    qkv = torch.randn(bs, (Hq + 2 * Hkv) * D, generator=g).to(dtype)
    cache = ops.rope_cos_sin_cache(max(lens) + 3, 10000.0, D).to(dtype)
    pos, seq = torch.tensor(lens) - 1, torch.tensor(lens)
    ks, vs = (0.5, 2.0) if bytes_pool else (1.0, 1.0)

    dev = {n: t.to(DEV) for n, t in dict(kb=kb, vb=vb, qkv=qkv, cache=cache, table=table, loc=loc, pos=pos, seq=seq, rows=rows).items()}
    out = torch.full((bs, Hq * D), float("nan"), dtype=dtype, device=DEV)
    q, k, v = dev["qkv"].split([Hq * D, Hkv * D, Hkv * D], 1)
    _native.decode_small(out, q, k, v, dev["pos"], dev["cache"], dev["loc"], dev["kb"], dev["vb"], dev["table"], dev["rows"], dev["seq"],
                         D ** -0.5, max(lens), ks, vs)

    q, k, v = qkv.split([Hq * D, Hkv * D, Hkv * D], 1)
    q, k = ops.rotary_embedding(pos, q.clone(), k.clone(), D, cache, True)
    kb[loc] = (k.reshape(bs, Hkv, D) / ks).to(pool_type)
    vb[loc] = (v.reshape(bs, Hkv, D) / vs).to(pool_type)
    assert torch.equal(dev["kb"].cpu().view(torch.uint8), kb.view(torch.uint8)) and torch.equal(dev["vb"].cpu().view(torch.uint8), vb.view(torch.uint8))
    assert torch.equal(dev["qkv"].cpu(), qkv)
    attend = lambda values: ops.decode_attention(q.reshape(bs, Hq, D).float(), kb.float() * ks, values * vs, table, rows, seq, D ** -0.5)  # noqa: E731
    # (a byte pool's products are in fp16: its unit roundoff joins bf16's in the output)
    assert_attn_close(out.view(bs, Hq, D), attend(vb.float()), attend(vb.float().abs()), dtype, what=f"{dtype} {Hq}/{Hkv} x {D} {lens}",
                      units=2.0 if bytes_pool and dtype == torch.float16 else 1.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bytes_pool", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", [[300], [1000], [100, 400, 50, 200]])
def test_no_further_off_than_the_three_launches(dtype, bytes_pool, D, lens):
    """both round weights to the 16-bit type; the mean error over seeds and rows (the oracle's sums are fp32, 1e-7) is held to the general form's, a
    thousandth for the mean's own noise where the output's rounding is all there is"""
    from scratchpad_amd import _native
    Hq, Hkv, bs = 32, 8, len(lens)
    pool_type = torch.float8_e5m2 if bytes_pool else dtype
    cache = ops.rope_cos_sin_cache(max(lens), 10000.0, D).to(dtype).to(DEV)
    seq, rows, errors = torch.tensor(lens, device=DEV), torch.arange(bs, device=DEV), torch.zeros(2, dtype=torch.float64)
    for seed in range(6):
        g = torch.Generator(device=DEV).manual_seed(seed)
        kb, vb = (torch.randn(sum(lens), Hkv, D, generator=g, device=DEV).to(pool_type) for _ in range(2))
        perm, table, at = torch.randperm(sum(lens), generator=g, device=DEV), torch.zeros(bs, max(lens), dtype=torch.int32, device=DEV), 0
        for r, n in enumerate(lens):
            table[r, :n] = perm[at:at + n].int()
            at += n
        loc = table[rows, seq - 1].long()
        qkv, out = torch.randn(bs, (Hq + 2 * Hkv) * D, generator=g, device=DEV).to(dtype), torch.empty(2, bs, Hq, D, dtype=dtype, device=DEV)
        q, k, v = qkv.split([Hq * D, Hkv * D, Hkv * D], 1)
        _native.decode_small(out[0].view(bs, -1), q, k, v, seq - 1, cache, loc, kb, vb, table, rows, seq, D ** -0.5, max(lens))
        q, k = q.contiguous(), k.contiguous()
        _native.rotary_embedding(seq - 1, q, k, D, cache, True)
        ranges = _native.decode_ranges(Hq, Hkv, D, dtype, pool_type)
        ws = torch.empty(_native.decode_workspace_bytes(bs, Hq, D, max(lens), 64, 0, ranges), dtype=torch.uint8, device=DEV)
        plan = torch.empty(_native.decode_plan_bytes(bs, max(lens), 64, 0, ranges) // 4, dtype=torch.int32, device=DEV)
        _native.decode_plan(plan, seq, max(lens), 64, 0, ranges)
        _native.decode_attention(out[1], q.view(bs, Hq, D), kb, vb, table, rows, seq, D ** -0.5, 0.0, max(lens), 64, ws, None, plan, max_slots=0,
                                 ranges=ranges)
        want = ops.decode_attention(*(t.cpu() for t in (q.view(bs, Hq, D).float(), kb.float(), vb.float(), table, rows, seq)), D ** -0.5).double()
        errors += ((out.cpu().double() - want) ** 2).sum((1, 2, 3)) / (want ** 2).sum()
    small, general = errors.sqrt().tolist()
    assert small <= 1.001 * general, f"{small / general:.4f}"


def _steps(mr, n, steps, hook=False):
    """logits of `steps` decode steps of n requests of unequal lengths"""
    from scratchpad_amd.forward_info import ForwardMode, ModelWorkerBatch
    from scratchpad_amd.model_runner import TpModelWorker
    worker, calls = TpModelWorker(mr), []
    if hook:
        mr.model.model.layers[0].self_attn.attn.register_forward_hook(lambda *_: calls.append(1))
    gen = torch.Generator(device=mr.device).manual_seed(5)
    for layer in range(2):
        for buf in mr.token_to_kv_pool.get_kv_buffer(layer):
            buf.copy_(torch.randn(buf.shape, generator=gen, device=mr.device).to(buf.dtype))
    lens = torch.tensor([5, 17, 9][:n], device=mr.device)
    req = torch.arange(1, n + 1, device=mr.device)
    for i, row in enumerate(req.tolist()):
        mr.req_to_token_pool.req_to_token[row, :30] = torch.arange(1 + 30 * i, 31 + 30 * i, device=mr.device, dtype=torch.int32)
    out = []
    for s in range(steps):
        lens = lens + 1
        loc = mr.req_to_token_pool.req_to_token[req, lens - 1].long()
        batch = ModelWorkerBatch(bid=s, forward_mode=ForwardMode.DECODE, input_ids=torch.arange(3, 3 + n, device=mr.device) + s, req_pool_indices=req,
                                 seq_lens=lens, out_cache_loc=loc, seq_lens_sum=int(lens.sum()))
        out.append(worker.forward_batch_generation(batch)[0].next_token_logits.float().cpu())
    return torch.stack(out), calls


@pytest.mark.parametrize("graph", [None, [2, 4]])
def test_small_steps_of_a_model(graph, monkeypatch):
    """the model's small steps run the one launch, eagerly and replayed, and agree with the general form; a layer with a hook is called"""
    from scratchpad_amd import _native, attention
    from scratchpad_amd.model_runner import ModelConfig, ModelRunner, ServerArgs
    small = []
    real = _native.decode_small
    monkeypatch.setattr(_native, "decode_small", lambda *a, **k: (small.append(1), real(*a, **k)))

    def runner():
        cfg = ModelConfig(256, 512, 2, 4, 2, 640, context_len=60)
        mr = ModelRunner(cfg, ServerArgs(max_total_tokens=96, max_running_requests=3, disable_cuda_graph=graph is None, cuda_graph_bs=graph),
                         dtype=torch.bfloat16, seed=3, init_weights=True)
        return mr
    mr = runner()
    if graph:
        mr.init_cuda_graphs()
    assert mr.attn_backend.small_steps
    got, _ = _steps(mr, 3, 4)
    assert len(small) > 0
    hooked = runner()
    want_hook, calls = _steps(hooked, 3, 4, hook=True)          # eager: layer 0 by itself, layer 1 in one launch
    assert len(calls) == 4
    monkeypatch.setattr(attention.HipAttnBackend, "SMALL_MAX_ROWS", 0)
    mr = runner()
    if graph:
        mr.init_cuda_graphs()
    want, _ = _steps(mr, 3, 4)
    for x in (got, want_hook):
        # two orders of the same sums: a few roundings of 2^-9 through two layers
        assert float((x - want).norm() / want.norm()) < 0.01


# lengths of three requests, and whether the step is small, eagerly and replayed in the bucket of four (whose padded row holds one key): at the bounds
# 1280 and 1408 of heads of 64, past them, and back
WALK = [((400, 430, 450), True, True), ((401, 431, 451), False, True), ((440, 480, 487), False, True), ((441, 481, 488), False, False),
        ((5, 17, 9), True, True), ((700, 600, 600), False, False), ((6, 18, 10), True, True)]


@pytest.mark.parametrize("hooked", [None, 0, 1])
@pytest.mark.parametrize("graph", [None, [2, 4]])
def test_steps_cross_the_bound_of_keys(graph, hooked, monkeypatch):
    """a model's steps go from one form to the other and back as its requests grow, are served and start anew: which form ran, and that every
    step's logits are the general form's.  With a hook on a layer (there before the graphs are captured) that layer is called by itself: its
    plan is built once a step, under capture as a launch of the graph."""
    from scratchpad_amd import attention
    from scratchpad_amd.forward_info import ForwardMode, ModelWorkerBatch
    from scratchpad_amd.model_runner import ModelConfig, ModelRunner, ServerArgs, TpModelWorker

    def walk(hooked):
        cfg = ModelConfig(256, 512, 2, 4, 2, 640, context_len=800)
        mr = ModelRunner(cfg, ServerArgs(max_total_tokens=2500, max_running_requests=3, disable_cuda_graph=graph is None, cuda_graph_bs=graph),
                         dtype=torch.bfloat16, seed=3, init_weights=True)
        forms, calls, out = [], [], []
        if hooked is not None:
            mr.model.model.layers[hooked].self_attn.attn.register_forward_hook(lambda *_: calls.append(1))
        if graph:
            mr.init_cuda_graphs()

            class Noted:
                def __init__(self, graph, small):
                    self.graph, self.small = graph, small

                def replay(self):
                    forms.append(self.small)
                    self.graph.replay()
            runner = mr.graph_runner
            runner.graphs = {b: Noted(g, False) for b, g in runner.graphs.items()}
            runner.small_graphs = {b: (Noted(g, True), o) for b, (g, o) in runner.small_graphs.items()}
        gen = torch.Generator(device=mr.device).manual_seed(5)
        for layer in range(2):
            for buf in mr.token_to_kv_pool.get_kv_buffer(layer):
                buf.copy_(torch.randn(buf.shape, generator=gen, device=mr.device).to(buf.dtype))
        req = torch.arange(1, 4, device=mr.device)
        for i, row in enumerate(req.tolist()):
            mr.req_to_token_pool.req_to_token[row, :800] = torch.arange(1 + 800 * i, 801 + 800 * i, device=mr.device, dtype=torch.int32)
        worker = TpModelWorker(mr)
        for s, (lens, *_) in enumerate(WALK):
            seq = torch.tensor(lens, device=mr.device)
            batch = ModelWorkerBatch(bid=s, forward_mode=ForwardMode.DECODE, input_ids=torch.arange(3, 6, device=mr.device) + s, req_pool_indices=req,
                                     seq_lens=seq, out_cache_loc=mr.req_to_token_pool.req_to_token[req, seq - 1].long(), seq_lens_sum=sum(lens))
            out.append(worker.forward_batch_generation(batch)[0].next_token_logits.float().cpu())
            if not graph:
                forms.append(mr.attn_backend.small_step)
        return out, forms, calls

    got, forms, calls = walk(hooked)
    assert forms == [w[2 if graph else 1] for w in WALK] and (hooked is None) == (not calls)
    monkeypatch.setattr(attention.HipAttnBackend, "SMALL_MAX_ROWS", 0)
    want, general, _ = walk(None)
    assert not any(general)
    for s, (x, y) in enumerate(zip(got, want)):
        # two orders of the same sums: a few roundings of 2^-9 through two layers
        assert float((x - y).norm() / y.norm()) < 0.01, f"step {s}, {WALK[s]}"
