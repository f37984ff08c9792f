"""The work that users of this framework have it do, as cases that can be timed and compared.

Kinds of case, each through the classes that a serving program calls:

* ``llama``: one step of a Llama model through ModelRunner / TpModelWorker, from a scheduled batch to its logits - a decode
  step (HIP-graph replay, paged keys and values at scattered slots) or a batch of prompts (with or without a cached prefix);
* ``mixer`` / ``attention``: one layer of the recurrent and windowed or latent attention designs over its request state or
  cache, input projection to output projection, in prompt batches and in decode steps;
* ``experts``: a routed feed-forward layer, router to weighted sum.

The designs with routed experts are taken layer by layer and not as whole models because a 16-bit model's logits cannot be
compared over a chain of routers (one expert chosen otherwise is another result); every Llama case is a model of its own.
Widths, heads, states and expert counts are those of the repository's configurations and benchmark (``bench_hybrid.py``)."""
import math
import random
from types import SimpleNamespace

import torch

DEV = "cuda"
VOCAB = 128256
# (hidden, feed-forward, query heads, key/value heads, head size, layers run, tied head, llama3 rope scaling)
LLAMA = {"1b": (2048, 8192, 32, 8, 64, 16, True, True),        # Llama-3.2-1B, whole
         "8b": (4096, 14336, 32, 8, 128, 4, False, False)}     # Llama-3-8B, a stretch of its 32 equal layers
MIXERS = ("mamba2", "mlstm", "general_delta", "gated_delta", "head_delta", "hgrn2")
EXPERTS, TOP = 32, 4
EPS = 1e-5


# ------------------------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one user's chat: every token is one step of one row, nothing but weights and launches
        dict(name="chat token", kind="llama", model="1b", mode="decode", requests=1, tokens=300, prefix=0,
             dtype="bfloat16", kv="auto"),
        # a server's full batch at ragged contexts: the headline decode step
        dict(name="serving decode", kind="llama", model="8b", mode="decode", requests=256, tokens=546880, prefix=0,
             dtype="bfloat16", kv="auto"),
        # fewer, longer requests over a one-byte cache, a batch between two graph sizes
        dict(name="long fp8 decode", kind="llama", model="8b", mode="decode", requests=61, tokens=250009, prefix=0,
             dtype="bfloat16", kv="fp8_e5m2"),
        # time to first token of a full prefill batch
        dict(name="prompt batch", kind="llama", model="8b", mode="prompt", requests=8, tokens=16384, prefix=0,
             dtype="bfloat16", kv="auto"),
        # chunked prefill: portions of odd length behind cached prefixes
        dict(name="prompt portions", kind="llama", model="1b", mode="prompt", requests=3, tokens=777, prefix=1500,
             dtype="float16", kv="auto"),
        # prompts through the state-space, matrix-memory and delta-rule layers of the hybrid designs
        dict(name="mamba2 prompts", kind="mixer", mixer="mamba2", width=2048, mode="prompt", requests=8, tokens=4096),
        dict(name="mlstm prompts", kind="mixer", mixer="mlstm", width=2048, mode="prompt", requests=5, tokens=3001),
        dict(name="gated delta prompts", kind="mixer", mixer="gated_delta", width=2048, mode="prompt", requests=8, tokens=4096),
        # the same layers one token per request
        dict(name="general delta decode", kind="mixer", mixer="general_delta", width=1024, mode="decode", requests=16, tokens=16),
        # windowed attention with pooled blocks over long prompts
        dict(name="window prompts", kind="attention", layer="window", width=2048, mode="prompt", requests=4, tokens=4096, prefix=0),
        # routed experts: a prompt batch, and a small decode step that touches most experts once
        dict(name="experts prompts", kind="experts", act="silu", width=2048, tokens=4096),
        dict(name="experts decode", kind="experts", act="clamped", width=2048, tokens=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    case = dict(rng.choice(listed()))
    del case["name"]
    if case["kind"] == "llama":
        case["model"] = rng.choice(("1b", "8b"))
        case["dtype"] = rng.choice(("bfloat16", "bfloat16", "float16"))
        if case["mode"] == "decode":
            case["requests"] = _log(rng, 1, 256)
            case["tokens"] = min(case["requests"] * _log(rng, 64, 4096), 546880 if case["model"] == "8b" else 260000)
            case["kv"] = rng.choice(("auto", "auto", "fp8_e5m2"))
        else:
            case["tokens"] = _log(rng, 17, 12000)
            case["requests"] = min(_log(rng, 1, 16), max(1, case["tokens"] // 16))
            case["prefix"] = rng.choice((0, _log(rng, 16, 2048)))
    elif case["kind"] == "experts":
        case["act"] = rng.choice(("silu", "clamped"))
        case["width"] = rng.choice((1024, 2048))
        case["tokens"] = _log(rng, 1, 4096)
    else:
        case["width"] = rng.choice((1024, 2048))
        case["mode"] = rng.choice(("prompt", "prompt", "decode"))
        if case["kind"] == "mixer":
            case["mixer"] = rng.choice(MIXERS)
        else:
            case["layer"] = rng.choice(("window", "latent"))
            case["prefix"] = _log(rng, 16, 4096) if case["mode"] == "decode" else rng.choice((0, _log(rng, 16, 2048)))
        if case["mode"] == "decode":
            case["requests"] = case["tokens"] = _log(rng, 1, 64)
        else:
            case["tokens"] = _log(rng, 65, 4096)
            case["requests"] = min(_log(rng, 1, 16), max(1, case["tokens"] // 16))
    return case


def _lengths(n, total, low=1):
    """`n` unequal lengths of at least `low` that sum to `total` (a case's own: the same for every seed)"""
    r = random.Random(total * 1009 + n)
    share = [r.uniform(1.0, 32.0) for _ in range(n)]
    free = total - low * n
    out = [low + int(free * s / sum(share)) for s in share]
    for i in range(total - sum(out)):
        out[i % n] += 1
    return out


# ------------------------------------------------------------------------------------------------------------ shared
def _randn(gen, *shape, std=1.0, dtype=torch.bfloat16):
    out = torch.empty(shape, dtype=dtype, device=DEV)
    return out.normal_(0.0, std, generator=gen)


def _weights(module, gen, matrix_std=None):
    """random weights of a trained layer's scale: matrices that keep the variance, decays and gates inside their range"""
    for name, p in module.named_parameters():
        leaf = name.rsplit(".", 1)[-1]
        if "norm" in name:
            p.data.uniform_(0.7, 1.3, generator=gen)
        elif leaf in ("A_log", "dt_bias"):
            p.data.normal_(-1.0, 0.5, generator=gen)
        elif leaf == "gates_bias":
            p.data.normal_(1.0, 1.0, generator=gen)
        elif leaf == "lower":
            p.data.uniform_(0.0, 0.5, generator=gen)
        elif leaf == "D":
            p.data.normal_(1.0, 0.3, generator=gen)
        elif leaf == "conv":
            p.data.normal_(0.0, 0.5, generator=gen)
        elif p.dim() >= 2:
            fan_in = p.shape[0] if leaf in ("w2t", "a2t", "g2t") else p.shape[-1]
            p.data.normal_(0.0, matrix_std or fan_in ** -0.5, generator=gen)
        else:
            p.data.normal_(0.0, 0.1, generator=gen)


def _ints(values, dtype=torch.int64):
    return torch.tensor(values, dtype=dtype).to(DEV)


def _batch(case, lens, held, slots_of, pools):
    """the step's ForwardBatch of a layer case: request i holds held[i] tokens and brings lens[i]"""
    from scratchpad_amd.attention import SequenceBackend
    from scratchpad_amd.forward_info import ForwardBatch, ForwardMode
    n = len(lens)
    seq = [p + e for p, e in zip(held, lens)]
    backend = SequenceBackend(SimpleNamespace(device=DEV, model_config=SimpleNamespace(context_len=max(seq) + 4)))
    table = torch.zeros((n + 1, max(seq) + 4), dtype=torch.int32, device=DEV)
    new = []
    for i, s in enumerate(slots_of):
        table[i + 1, :seq[i]] = s.to(torch.int32)
        new.append(s[held[i]:])
    fb = ForwardBatch(
        forward_mode=ForwardMode.DECODE if case["mode"] == "decode" else ForwardMode.EXTEND, batch_size=n,
        input_ids=torch.zeros(sum(lens), dtype=torch.int64, device=DEV), req_pool_indices=_ints(range(1, n + 1)),
        seq_lens=_ints(seq), out_cache_loc=torch.cat(new), seq_lens_sum=sum(seq),
        positions=_ints([p + t for p, e in zip(held, lens) for t in range(e)]),
        req_to_token_pool=SimpleNamespace(req_to_token=table), attn_backend=backend, **pools)
    if case["mode"] != "decode":
        starts = [sum(lens[:i]) for i in range(n)]
        fb.extend_num_tokens = sum(lens)
        fb.extend_seq_lens, fb.extend_prefix_lens = _ints(lens, torch.int32), _ints(held, torch.int32)
        fb.extend_start_loc = _ints(starts, torch.int32)
        fb.extend_seq_lens_cpu, fb.extend_prefix_lens_cpu = list(lens), list(held)
    return fb


def _slots(gen, lens):
    """scattered cache slots (1-based; slot 0 is the pool's dummy), one tensor per request"""
    return list((torch.randperm(sum(lens), generator=gen, device=DEV) + 1).split(list(lens)))


# ------------------------------------------------------------------------------------------------------------ llama
def _llama_lens(case):
    """(tokens held, tokens brought) per request"""
    if case["mode"] == "decode":
        return [n - 1 for n in _lengths(case["requests"], case["tokens"], 2)], [1] * case["requests"]
    return [case["prefix"] + 7 * i if case["prefix"] else 0 for i in range(case["requests"])], \
        _lengths(case["requests"], case["tokens"])


def _prepare_llama(case, seed):
    from scratchpad_amd.forward_info import ForwardMode
    from scratchpad_amd.model_runner import ModelConfig, ModelRunner, ServerArgs, TpModelWorker
    from scratchpad_amd.schedule_batch import Req, ScheduleBatch
    gen = torch.Generator(device=DEV).manual_seed(seed)
    host = random.Random(seed)
    held, lens = _llama_lens(case)
    n, total = len(lens), sum(held) + sum(lens)
    layers = LLAMA[case["model"]][5]
    context = max(p + e for p, e in zip(held, lens)) + 8
    cfg = (ModelConfig.llama32_1b if case["model"] == "1b" else ModelConfig.llama3_8b)(context)
    cfg.num_hidden_layers = layers
    bucket = next(b for b in [1, 2, 4, 8] + list(range(16, 257, 8)) if b >= n) if n <= 256 else n
    args = ServerArgs(max_total_tokens=total + 64, max_running_requests=max(n, bucket), cuda_graph_max_bs=bucket,
                      cuda_graph_bs=[bucket], kv_cache_dtype=case["kv"])
    mr = ModelRunner(cfg, args, dtype=getattr(torch, case["dtype"]), seed=seed, init_weights=False)
    _weights(mr.model, gen, 0.02)
    for name, p in mr.model.named_parameters():
        # a stream that each layer adds a part to, as in a trained model: with 0.02 throughout, every layer drowns the ones
        # before it and the 16-bit roundings with them
        if "embed_tokens" in name:
            p.data.normal_(0.0, 1.0, generator=gen)
        elif "o_proj" in name or "down_proj" in name:
            p.data.mul_((2 * layers) ** -0.5)
    if case["mode"] == "decode":
        mr.init_cuda_graphs()
    pool, alloc = mr.token_to_kv_pool, mr.token_to_kv_pool_allocator
    kv = [pool.get_kv_buffer(l) for l in range(layers)]
    for pair in kv:
        for buf in pair:
            if buf.dtype == torch.float8_e5m2:
                buf.copy_(_randn(gen, *buf.shape, std=0.5).to(torch.float8_e5m2))
            else:
                buf.normal_(0.0, 0.5, generator=gen)
    # the free list of a server that has run for a while: slots in no order
    alloc.free_slots = torch.randperm(alloc.size, generator=gen, device=DEV) + 1
    ids = [[host.randrange(VOCAB) for _ in range(p + e)] for p, e in zip(held, lens)]
    if case["mode"] == "decode":
        batch = ScheduleBatch([Req(str(i), "", [], None) for i in range(n)], mr.req_to_token_pool, alloc, model_config=cfg,
                              device=mr.device)
        rows = batch.alloc_req_slots(n)
        slots = alloc.alloc(sum(held)).split(held)
        for row, s in zip(rows, slots):
            mr.req_to_token_pool.req_to_token[row, :s.shape[0]] = s.to(torch.int32)
        batch.req_pool_indices, batch.seq_lens, batch.seq_lens_sum = _ints(rows), _ints(held), sum(held)
        batch.output_ids = _ints([r[-1] for r in ids])
        batch.forward_mode = ForwardMode.DECODE
        batch.prepare_for_decode()
    else:
        reqs = []
        for i in range(n):
            r = Req(str(i), "", ids[i], None)
            r.fill_ids = list(ids[i])
            r.prefix_indices = alloc.alloc(held[i]) if held[i] else torch.empty(0, dtype=torch.int64, device=DEV)
            reqs.append(r)
        batch = ScheduleBatch(reqs, mr.req_to_token_pool, alloc, model_config=cfg, device=mr.device)
        batch.prepare_for_extend()
    torch.cuda.synchronize()
    return SimpleNamespace(case=case, runner=mr, worker=TpModelWorker(mr), batch=batch.get_model_worker_batch(), kv=kv)


def _run_llama(s):
    out, _ = s.worker.forward_batch_generation(s.batch, skip_sample=True)
    return {"logits": out.next_token_logits, "last layer's keys": s.kv[-1][0], "last layer's values": s.kv[-1][1]}


def _llama_params(model):
    hidden, ff, hq, hk, d, layers, _, _ = LLAMA[model]
    return layers * (hidden * d * (2 * hq + 2 * hk) + 3 * hidden * ff)


def _work_llama(case):
    hidden, ff, hq, hk, d, layers, _, _ = LLAMA[case["model"]]
    held, lens = _llama_lens(case)
    n, t = len(lens), sum(lens)
    row = layers * 2 * hk * d * (1 if case["kv"] == "fp8_e5m2" else 2)
    pairs = sum(e * p + e * (e + 1) // 2 for p, e in zip(held, lens))
    return {"bytes": 2 * _llama_params(case["model"]) + 2 * VOCAB * hidden + 2 * t * hidden + (sum(held) + t) * row + 4 * n * VOCAB,
            "flops": 2 * t * _llama_params(case["model"]) + 2 * n * VOCAB * hidden + layers * 4 * hq * d * pairs}


def _rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _exact_llama(case, seed):
    s = _prepare_llama(case, seed)
    hidden, ff, hq, hk, d, layers, tied, scaled = LLAMA[case["model"]]
    held, lens = _llama_lens(case)
    w = dict(s.runner.model.named_parameters())
    table, b = s.runner.req_to_token_pool.req_to_token, s.batch
    rows = [table[r, :p + e].long() for r, p, e in zip(b.req_pool_indices.tolist(), held, lens)]
    freq = 500000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    if scaled:        # the llama3 rule: long waves slowed 32-fold, a blend between the two bounds
        wave = 2 * math.pi / freq
        mix = (8192 / wave - 1.0) / (4.0 - 1.0)
        freq = torch.where(wave < 8192 / 4.0, freq, torch.where(wave > 8192 / 1.0, freq / 32, (1 - mix) * freq / 32 + mix * freq))
    pos = torch.cat([torch.arange(p, p + e, device=DEV) for p, e in zip(held, lens)]).double()
    cos, sin = torch.cos(pos[:, None] * freq)[:, None], torch.sin(pos[:, None] * freq)[:, None]

    def turn(x):
        u, v = x[..., :d // 2], x[..., d // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

    x = w["model.embed_tokens.weight"].data[b.input_ids].double()
    t = x.shape[0]
    for l in range(layers):
        p = f"model.layers.{l}."
        mat = lambda name: w[p + name + ".weight"].data.double()  # noqa: E731
        qkv = (_rms(x) * mat("input_layernorm")) @ mat("self_attn.qkv_proj").t()
        q, k, v = (y.reshape(t, -1, d) for y in qkv.split([hq * d, hk * d, hk * d], 1))
        q, k = turn(q), turn(k)
        if case["kv"] == "fp8_e5m2":        # what a cache of one byte holds of the step's own rows
            k, v = (y.float().to(torch.float8_e5m2).double() for y in (k, v))
        o, at = torch.empty_like(q), 0
        for r, held_i, e in zip(rows, held, lens):
            kk = torch.cat([s.kv[l][0][r[:held_i]].double(), k[at:at + e]])
            vv = torch.cat([s.kv[l][1][r[:held_i]].double(), v[at:at + e]])
            seen = torch.arange(held_i + e, device=DEV)[None] <= torch.arange(held_i, held_i + e, device=DEV)[:, None]
            for g in range(hk):
                qq = q[at:at + e, g * hq // hk:(g + 1) * hq // hk].transpose(0, 1)
                sc = (qq @ kk[:, g].t().contiguous()) * d ** -0.5
                o[at:at + e, g * hq // hk:(g + 1) * hq // hk] = (
                    torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ vv[:, g].contiguous()).transpose(0, 1)
            at += e
        x = x + o.reshape(t, -1) @ mat("self_attn.o_proj").t()
        g, u = ((_rms(x) * mat("post_attention_layernorm")) @ mat("mlp.gate_up_proj").t()).split(ff, 1)
        x = x + (torch.nn.functional.silu(g) * u) @ mat("mlp.down_proj").t()
    last = torch.tensor(lens).cumsum(0).to(DEV) - 1
    head = w["model.embed_tokens.weight" if tied else "lm_head.weight"].data[:VOCAB]
    return {"logits": (_rms(x[last]) * w["model.norm.weight"].data.double()) @ head.double().t(), "last layer's keys": None,
            "last layer's values": None}


# ------------------------------------------------------------------------------------------------------------ mixers
def _mixer(kind, w):
    """(module, its state's shapes), heads and states as in the repository's benchmark configurations at this width"""
    from scratchpad_amd import recurrent as R
    bf = torch.bfloat16
    if kind == "mamba2":
        return R.Mamba2Mixer(w, 2 * w // 64, 64, 128, 8, 4, 8, 0, EPS, bf), R.Mamba2Mixer.state_shapes(2 * w // 64, 64, 128, 8, 4)
    if kind == "mlstm":
        return R.MLSTMMixer(w, w // 128, 128, 128, 15.0, 0, EPS, bf), R.MLSTMMixer.state_shapes(w // 128, 128, 128)
    if kind == "general_delta":
        return R.GeneralDeltaMixer(w, w // 64, 64, 64, EPS, layer_id=0, dtype=bf), R.GeneralDeltaMixer.state_shapes(w // 64, 64)
    if kind == "gated_delta":
        a = (w // 128, w // 256, 128, 128, 4)
        return R.GatedDeltaMixer(w, *a, 64, 64, EPS, layer_id=0, dtype=bf), R.GatedDeltaMixer.state_shapes(*a)
    if kind == "head_delta":
        a = (w // 128, w // 256, 128, 128, 4)
        return R.HeadDeltaMixer(w, *a, EPS, layer_id=0, dtype=bf), R.HeadDeltaMixer.state_shapes(*a)
    return R.HGRN2Mixer(w, w // 256, 128, 128, EPS, layer_id=0, dtype=bf), R.HGRN2Mixer.state_shapes(w // 256, 128, 128)


def _prepare_mixer(case, seed):
    from scratchpad_amd.pool import RecurrentStatePool
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n, decode = case["requests"], case["mode"] == "decode"
    lens = [1] * n if decode else _lengths(n, case["tokens"])
    held = [9 + i for i in range(n)] if decode else [0] * n
    with torch.device(DEV):
        mixer, shapes = _mixer(case["mixer"], case["width"])
    _weights(mixer, gen)
    pool = RecurrentStatePool(n + 1, case["width"], {}, DEV, shift_layers=[], named={0: shapes})
    if decode:        # what a request's earlier tokens have left (a new prompt starts from the initial state)
        for name in sorted(shapes):
            pool.state(0, name)[1:].normal_(0.0, 0.5, generator=gen)
    fb = _batch(case, lens, held, [torch.arange(1, p + e + 1, device=DEV) for p, e in zip(held, lens)], {"state_pool": pool})
    return SimpleNamespace(case=case, mixer=mixer, h=_randn(gen, sum(lens), case["width"]), fb=fb, lens=lens,
                           state={name: pool.state(0, name) for name in shapes})


def _run_mixer(s):
    s.fb.attn_backend.init_forward_metadata(s.fb)
    return {"y": s.mixer(s.h, s.fb), **{name: t[1:] for name, t in s.state.items()}}


def _work_mixer(case):
    w, n, t = case["width"], case["requests"], case["tokens"]
    kind = case["mixer"]
    # columns of the input projection, elements of all heads' states, width of the mixer's inner result, flops per state element
    cols, state, inner, per = {"mamba2": (4 * w + 2048 + w // 32, 2 * w // 64 * 64 * 128, 2 * w, 4),
                               "mlstm": (4 * w + w // 64, w * 128, w, 4),
                               "general_delta": (5 * w + 64, w * 64, w, 9),
                               "gated_delta": (2 * w + w // 128 + 128, w * 128, w, 7),
                               "head_delta": (3 * w + w // 64, w * 128, w, 7),
                               "hgrn2": (3 * w // 2, w // 2 * 128, w // 2, 5)}[kind]
    weights = w * (cols + inner) + (64 * 2 * w if kind in ("gated_delta", "general_delta") else 0)
    return {"bytes": 2 * weights + 4 * t * w + 4 * n * state * (2 if case["mode"] == "decode" else 1),
            "flops": 2 * t * weights + per * t * state}


def _scan(lens, state, step, *inputs):
    """64-bit recurrence over packed requests: step(state, *rows) -> (state, out row) for all requests side by side"""
    starts = [sum(lens[:i]) for i in range(len(lens))]
    out = None
    for t in range(max(lens)):
        live = [i for i, n in enumerate(lens) if t < n]
        at = _ints([starts[i] for i in live]) + t
        now = state if len(live) == len(lens) else {k: v[_ints(live)] for k, v in state.items()}
        now, o = step(now, *(x[at] for x in inputs))
        out = torch.zeros((sum(lens),) + tuple(o.shape[1:]), dtype=o.dtype, device=DEV) if out is None else out
        out[at] = o
        if len(live) == len(lens):
            state = now
        else:
            for k in state:
                state[k][_ints(live)] = now[k]
    return out, state


def _conv(u, weight, bias, state, lens):
    """(silu of the causal convolution, the latest taps - 1 inputs per request); state [requests, taps - 1, channels]"""
    taps, parts, last, at = weight.shape[1], [], [], 0
    for i, n in enumerate(lens):
        pad = torch.cat([state[i], u[at:at + n]])
        parts.append(sum(pad[j:j + n] * weight[:, j] for j in range(taps)) + bias)
        last.append(pad[n:])
        at += n
    return torch.nn.functional.silu(torch.cat(parts)), torch.stack(last)


def _exact_mixer(case, seed):
    F = torch.nn.functional
    s = _prepare_mixer(case, seed)
    m, lens, kind, h = s.mixer, s.lens, case["mixer"], s.h.double()
    w = {k: p.data.double() for k, p in m.named_parameters()}
    t, n = h.shape[0], len(lens)
    st = {k: (v[1:].double() if case["mode"] == "decode" else torch.zeros_like(v[1:], dtype=torch.float64))
          for k, v in s.state.items()}
    H = m.heads
    outer = lambda a, b: a[..., :, None] * b[..., None, :]  # noqa: E731
    read = lambda S, x: (S * x[..., :, None]).sum(-2)       # noqa: E731  S^T x
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    if kind == "mamba2":
        G, N, V, inner = m.groups, m.state, m.vdim, H * m.vdim
        zx = h @ w["in_proj"].t()
        xbc, st["conv"] = _conv(zx[:, inner:], w["conv"], w["conv_bias"], st["conv"], lens)
        x, B, C = xbc[:, :inner].view(t, H, V), xbc[:, inner:inner + G * N].view(t, G, N), xbc[:, inner + G * N:].view(t, G, N)
        B, C = (y.repeat_interleave(H // G, 1) for y in (B, C))
        dt = F.softplus(h @ w["dt_proj"].t() + w["dt_bias"])

        def step(S, x, B, C, dt):
            new = S["ssm"] * torch.exp(-torch.exp(w["A_log"]) * dt)[..., None, None] + outer(B * dt[..., None], x)
            return {"ssm": new}, read(new, C) + w["D"][:, None] * x
        y, new = _scan(lens, {"ssm": st["ssm"]}, step, x, B, C, dt)
        y = _rms((y.reshape(t, inner) * F.silu(zx[:, :inner])).view(t, m.norm_groups, -1)).reshape(t, inner) * w["norm"]
        return {"y": y @ w["o"].t(), "ssm": new["ssm"], "conv": st["conv"]}
    if kind == "mlstm":
        D, V = m.dim, m.vdim
        q, k, v, g = (h @ w["qkvg"].t()).split([H * D, H * D, H * V, H * V], 1)
        gates = m.cap * torch.tanh((h @ w["gates"].t() + w["gates_bias"]) / m.cap)
        ig, fg = gates[:, :H], F.logsigmoid(gates[:, H:])

        def step(S, q, k, v, ig, fg):
            top = torch.maximum(fg + S["m"], ig)
            keep, take = torch.exp(fg + S["m"] - top), torch.exp(ig - top)
            mem = S["S"] * keep[..., None, None] + outer(k * take[..., None], v)
            nrm = S["n"] * keep[..., None] + k * take[..., None]
            den = torch.maximum((nrm * q).sum(-1).abs(), torch.exp(-top)) + 1e-6
            return {"S": mem, "n": nrm, "m": top}, read(mem, q) / den[..., None]
        y, new = _scan(lens, st, step, q.reshape(t, H, D) * D ** -0.5, k.reshape(t, H, D), v.reshape(t, H, V), ig, fg)
        return {"y": (_rms(y).reshape(t, -1) * w["norm"] * torch.sigmoid(g)) @ w["o"].t(), **new}
    if kind == "general_delta":
        D, r = m.dim, m.rank
        a = h @ w["in_proj"].t()
        rr, k, v, g, rem = (a[:, i * H * D:(i + 1) * H * D] for i in range(5))
        dec = torch.exp(-m.rate * torch.sigmoid(torch.tanh(a[:, 5 * H * D:5 * H * D + r]) @ w["w2t"] + w["w0"]))
        rem = torch.sigmoid(rem + w["a_bias"])

        def step(S, r, k, v, dec, rem):
            u = unit(k)
            new = S["S"] * dec[..., None] - outer(rem * u, read(S["S"], u)) + outer(k, v)
            return {"S": new}, read(new, r)
        y, new = _scan(lens, st, step, *(x.reshape(t, H, D) for x in (rr, k, v, dec, rem)))
        return {"y": (_rms(y).reshape(t, -1) * w["norm"] * torch.sigmoid(g)) @ w["o"].t(), **new}
    if kind == "hgrn2":
        D, V = m.dim, m.vdim
        q, f, v = (h @ w["in_proj"].t()).split([H * D, H * D, H * V], 1)
        f = w["lower"] + (1 - w["lower"]) * torch.sigmoid(f + w["f_bias"])

        def step(S, q, f, v):
            new = S["S"] * f[..., None] + outer(1 - f, v)
            return {"S": new}, read(new, q)
        y, new = _scan(lens, st, step, F.silu(q).reshape(t, H, D), f.reshape(t, H, D), v.reshape(t, H, V))
        return {"y": (_rms(y) * w["norm"]).reshape(t, -1) @ w["o"].t(), **new}
    # the two delta rules behind a convolution: a decay per key channel and head, or one per head
    G, D, V, c = m.kv_heads, m.dim, m.vdim, m.conv_rows
    a = h @ w["in_proj"].t()
    qkv, st["conv"] = _conv(a[:, :c], w["conv"], 0.0, st["conv"], lens)
    q, k = (qkv[:, i * G * D:(i + 1) * G * D].reshape(t, G, D).repeat_interleave(H // G, 1) for i in range(2))
    v = qkv[:, 2 * G * D:].reshape(t, H, V)
    if kind == "gated_delta":
        b, a1, g1 = a[:, c:].split([H, m.decay_rank, m.gate_rank], 1)
        dec = torch.exp(-torch.exp(w["A_log"])[:, None] * F.softplus(a1 @ w["a2t"] + w["dt_bias"]).view(t, H, D))
        gate = torch.sigmoid(g1 @ w["g2t"])
    else:
        b, al = (h @ w["gates"].t()).split(H, 1)
        dec = torch.exp(-torch.exp(w["A_log"]) * F.softplus(al + w["dt_bias"]))[..., None].expand(t, H, D)
        gate = F.silu(a[:, c:])

    def step(S, q, k, v, b, dec):
        kept = S["S"] * dec[..., None]
        new = kept + outer(k, b[..., None] * (v - read(kept, k)))
        return {"S": new}, read(new, q)
    y, new = _scan(lens, {"S": st["S"]}, step, unit(q) * D ** -0.5, unit(k), v, torch.sigmoid(b), dec)
    return {"y": ((_rms(y) * w["norm"]).reshape(t, -1) * gate) @ w["o"].t(), "S": new["S"], "conv": st["conv"]}


# ------------------------------------------------------------------------------------------------------------ attention
WINDOW, BLOCK, RANK, ROT = 512, 64, 512, 64


def _attention_lens(case):
    n = case["requests"]
    lens = [1] * n if case["mode"] == "decode" else _lengths(n, case["tokens"])
    return [case["prefix"] + 5 * i if case["prefix"] else 0 for i in range(n)], lens


def _prepare_attention(case, seed):
    from scratchpad_amd.pool import WindowKVPool
    gen = torch.Generator(device=DEV).manual_seed(seed)
    W, held_lens = case["width"], _attention_lens(case)
    held, lens = held_lens
    total = sum(held) + sum(lens)
    slots = _slots(gen, [p + e for p, e in zip(held, lens)])
    with torch.device(DEV):
        if case["layer"] == "window":
            from scratchpad_amd.sominex import SominexAttention
            m = {"heads": W // 128, "kv_heads": max(1, W // 512), "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                 "mask": {"size": WINDOW, "pool": BLOCK},
                 "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
            layer = SominexAttention(W, m, 0, EPS, torch.bfloat16)
            pool = WindowKVPool(total, torch.bfloat16, {0: (m["kv_heads"], 128, 128, True)}, DEV)
        else:
            from scratchpad_amd.kirenex import KirenexLatentAttention
            m = {"heads": W // 128, "dim": 128, "rot_dim": ROT, "vdim": 128, "kv_rank": RANK, "scale": (128 + ROT) ** -0.5,
                 "rot": {"base": 50000.0, "dims": ROT}}
            layer = KirenexLatentAttention(W, m, 0, EPS, torch.bfloat16)
            pool = WindowKVPool(total, torch.bfloat16, {}, DEV, latent={0: (RANK, ROT)})
    _weights(layer, gen)
    kbuf = pool.get_key_buffer(0)
    kbuf[1:].normal_(0.0, 1.0, generator=gen)
    state = [kbuf]
    if case["layer"] == "window":
        vbuf, (kp, vp) = pool.get_value_buffer(0), pool.get_pooled_buffers(0)
        vbuf[1:].normal_(0.0, 1.0, generator=gen)
        state += [vbuf, kp, vp]
        for s, p in zip(slots, held):        # the blocks that the cached tokens have completed
            whole = p // BLOCK
            if whole:
                for buf, means in ((kbuf, kp), (vbuf, vp)):
                    rows = buf[s[:whole * BLOCK]].float().view(whole, BLOCK, -1).mean(1)
                    means[s[BLOCK - 1:whole * BLOCK:BLOCK]] = rows.to(torch.bfloat16)
    fb = _batch(case, lens, held, slots, {"token_to_kv_pool": pool})
    return SimpleNamespace(case=case, layer=layer, m=m, h=_randn(gen, sum(lens), W), fb=fb, held=held, lens=lens,
                           slots=slots, state=state)


def _run_attention(s):
    s.fb.attn_backend.init_forward_metadata(s.fb)
    return [s.layer(s.fb.positions, s.h, s.fb)] + s.state


def _seen(case, p, e):
    """(query, key or block) pairs, rows read and rows written of a request"""
    if case["layer"] == "latent":
        return e * p + e * (e + 1) // 2, p + e, e
    pairs = sum(min(i + 1, WINDOW) + max(0, i - WINDOW + 1) // BLOCK for i in range(p, p + e))
    return pairs, min(p + e, WINDOW + e) + max(0, p + e - WINDOW) // BLOCK, e + (p + e) // BLOCK - p // BLOCK


def _work_attention(case):
    w = case["width"]
    held, lens = _attention_lens(case)
    t = sum(lens)
    seen = [_seen(case, p, e) for p, e in zip(held, lens)]
    if case["layer"] == "window":
        weights, row, per_pair = w * (w + w // 2 + w), 2 * max(1, w // 512) * 128, 2 * 256 * (w // 128)
    else:
        H = w // 128
        weights, row = w * (H * (128 + ROT) + RANK + ROT + w + w) + 2 * w * RANK, RANK + ROT
        per_pair = 2 * H * (2 * RANK + ROT)
    return {"bytes": 2 * weights + 4 * t * w + 2 * row * sum(r + x for _, r, x in seen),
            "flops": 2 * t * weights + per_pair * sum(p for p, _, _ in seen)}


def _turn(x, rotary, pos, adjacent):
    """x [T, heads, n]: the first dims coordinates rotated, as neighbours or as halves"""
    dims = rotary.dims
    ang = pos[:, None] * rotary.freq.double()[None]
    c, s = (torch.cos(ang) * rotary.magnitude)[:, None], (torch.sin(ang) * rotary.magnitude)[:, None]
    out = x.clone()
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if adjacent else (slice(0, dims // 2), slice(dims // 2, dims))
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _exact_attention(case, seed):
    s = _prepare_attention(case, seed)
    layer, m, h, pos = s.layer, s.m, s.h.double(), s.fb.positions.double()
    w = {k: p.data.double() for k, p in layer.named_parameters()}
    state = [t.double() for t in s.state]
    t, H = h.shape[0], m["heads"]
    loc, at = s.fb.out_cache_loc, 0
    if case["layer"] == "window":
        G, D = m["kv_heads"], 128
        q, k, v = (x.reshape(t, -1, D) for x in (h @ w["qkv"].t()).split([H * D, G * D, G * D], 1))
        q, k = _turn(q, layer.rotary, pos, False), _turn(k, layer.rotary, pos, False)
        kb, vb, kp, vp = state
        kb[loc], vb[loc] = k.reshape(t, -1), _rms(v).reshape(t, -1)
        o = torch.empty(t, H, D, dtype=torch.float64, device=DEV)
        for sl, p, e in zip(s.slots, s.held, s.lens):
            whole = (p + e) // BLOCK
            for b in range(p // BLOCK, whole):
                rows = sl[b * BLOCK:(b + 1) * BLOCK]
                kp[rows[-1]], vp[rows[-1]] = kb[rows].mean(0), vb[rows].mean(0)
            ends = sl[BLOCK - 1:whole * BLOCK:BLOCK]
            keys, vals = (torch.cat([x[sl], y[ends]]).view(-1, G, D) for x, y in ((kb, kp), (vb, vp)))
            i, j = torch.arange(p, p + e, device=DEV)[:, None], torch.arange(p + e, device=DEV)[None]
            blocks = torch.arange(whole, device=DEV)[None] * BLOCK + BLOCK - 1 <= i - WINDOW
            seen = torch.cat([(j <= i) & (i - j < WINDOW), blocks], 1)
            for n in range(H):
                g = n // (H // G)
                sc = (q[at:at + e, n] @ keys[:, g].t()) * m["scale"]
                o[at:at + e, n] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ vals[:, g]
            at += e
        return [o.reshape(t, -1) @ w["o"].t()] + state
    D, C, R = m["dim"], m["kv_rank"], m["rot_dim"]
    q, dkv, gate = (h @ w["in_proj"].t()).split([H * (D + R), C + R, H * 128], 1)
    q = q.reshape(t, H, D + R)
    q_rot = _turn(q[..., D:], layer.rotary, pos, True)
    pool = state[0]
    pool[loc] = torch.cat([_rms(dkv[:, :C]) * w["latent_norm"], _turn(dkv[:, None, C:], layer.rotary, pos, True)[:, 0]], 1)
    o = torch.empty(t, H, 128, dtype=torch.float64, device=DEV)
    for sl, p, e in zip(s.slots, s.held, s.lens):
        rows = pool[sl]
        seen = torch.arange(p + e, device=DEV)[None] <= torch.arange(p, p + e, device=DEV)[:, None]
        for n in range(H):
            sc = ((q[at:at + e, n, :D] @ w["uk_t"][n].t()) @ rows[:, :C].t() + q_rot[at:at + e, n] @ rows[:, C:].t()) * m["scale"]
            o[at:at + e, n] = (torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ rows[:, :C]) @ w["uv"][n].t()
        at += e
    return [(o.reshape(t, -1) * torch.sigmoid(gate)) @ w["o"].t()] + state


# ------------------------------------------------------------------------------------------------------------ experts
def _prepare_experts(case, seed):
    from scratchpad_amd import moe
    gen = torch.Generator(device=DEV).manual_seed(seed)
    W = case["width"]
    with torch.device(DEV):
        if case["act"] == "silu":
            layer = moe.SoftmaxMoE(W, EXPERTS, TOP, W // 2, 2.5, torch.bfloat16)
        else:
            layer = moe.ChosenSoftmaxMoE(W, EXPERTS, TOP, W // 2, 7.0, torch.bfloat16)
    _weights(layer, gen)
    return SimpleNamespace(case=case, layer=layer, x=_randn(gen, case["tokens"], W))


def _work_experts(case):
    w, t = case["width"], case["tokens"]
    one = 3 * w * (w // 2)
    used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** t)        # experts that some token of the step is expected to choose
    return {"bytes": 2 * one * used + 4 * EXPERTS * w + 4 * t * w, "flops": 2 * t * (TOP * one + EXPERTS * w)}


def _exact_experts(case, seed):
    s = _prepare_experts(case, seed)
    w = {k: p.data for k, p in s.layer.named_parameters()}
    x, ff = s.x.double(), case["width"] // 2
    score = x @ w["router.weight"].double().t()
    if case["act"] == "silu":
        val, ids = torch.topk(torch.softmax(score, -1), TOP)
        val = val * 2.5
    else:
        val, ids = torch.topk(score + w["router.bias"].double(), TOP)
        val = torch.softmax(val, -1)
    y = torch.zeros_like(x)
    for e in range(EXPERTS):
        tok, nth = torch.nonzero(ids == e, as_tuple=True)
        g, u = (x[tok] @ w["experts.gate_up"][e].double().t()).split(ff, 1)
        if case["act"] == "silu":
            a = torch.nn.functional.silu(g) * u
        else:
            g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
            a = g * torch.sigmoid(1.702 * g) * (u + 1)
        y.index_add_(0, tok, (a @ w["experts.down"][e].double().t()) * val[tok, nth][:, None])
    return y


# ------------------------------------------------------------------------------------------------------------ the file's uses
def prepare(case, seed):
    return {"llama": _prepare_llama, "mixer": _prepare_mixer, "attention": _prepare_attention,
            "experts": _prepare_experts}[case["kind"]](case, seed)


@torch.no_grad()
def run(state):
    kind = state.case["kind"]
    if kind == "experts":
        return state.layer(state.x)
    return {"llama": _run_llama, "mixer": _run_mixer, "attention": _run_attention}[kind](state)


def work(case):
    return {"llama": _work_llama, "mixer": _work_mixer, "attention": _work_attention,
            "experts": _work_experts}[case["kind"]](case)


def tolerance(case):
    """about four times the error against 64 bits that the listed cases show: 0.009 - 0.011 for a bf16 model's logits over its
    layers, 0.0014 in fp16; 0.0055 for one bf16 layer (at most 0.0034 for the fp32 state it leaves)"""
    if case["kind"] == "llama":
        return {"rel": 0.006, "max": 0.15} if case["dtype"] == "float16" and case["kv"] == "auto" else {"rel": 0.03, "max": 0.5}
    return {"rel": 0.02, "max": 0.5}


@torch.no_grad()
def exact(case, seed):
    return {"llama": _exact_llama, "mixer": _exact_mixer, "attention": _exact_attention,
            "experts": _exact_experts}[case["kind"]](case, seed)
