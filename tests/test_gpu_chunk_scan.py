"""The recurrences that run a chunk of 64 tokens at a time (bf16 rows, several tokens per request): mLSTM and Mamba-2 at the head
sizes the matrix form takes, requests whose lengths lie around the chunk's edges, from an empty and from a held state, against the
token-by-token recurrence in 64 bits.  What is fp32 is held to fp32: the inputs are exact, every product enters an fp32 sum, so the
states and Mamba-2's output differ from the 64-bit ones by accumulated fp32 roundings only - 64 + D additions and one exponential per
chunk, 2e-5 of the largest value being ten times that."""
import pytest
import torch

from tests.test_gpu_toredra_kernels import DEV, announce, seq_extend

pytestmark = pytest.mark.gpu
LENS = [[1], [63, 64, 65], [128, 1, 17, 200], [16, 48, 130, 2, 3]]


def near(got, want, bar):
    assert torch.isfinite(got).all()
    err = (got.double() - want).abs().max() / want.abs().max()
    assert err <= bar, f"{err:.2e} > {bar:.0e}"


def slots_of(lens):
    return [2 * i + 1 for i in range(len(lens))]


@pytest.mark.parametrize("lens", LENS, ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,D,Dv", [(3, 128, 128), (2, 128, 64), (2, 64, 128), (5, 64, 64)])
def test_mlstm_chunks(lens, H, D, Dv):
    from scratchpad_amd import _native
    announce("mlstm chunks", lens, H, D, Dv)
    g = torch.Generator(device=DEV).manual_seed(3)
    T, slots, cap, eps = sum(lens), slots_of(lens), 15.0, 1e-5
    n_slots = 2 * len(lens) + 1
    S = torch.full((n_slots, H, D, Dv), float("nan"), device=DEV)
    n, m = torch.full((n_slots, H, D), float("nan"), device=DEV), torch.full((n_slots, H), float("nan"), device=DEV)
    nw = torch.rand(H * Dv, generator=g, device=DEV) + 0.5
    ref = {s: (torch.zeros(H, D, Dv, dtype=torch.float64, device=DEV), torch.zeros(H, D, dtype=torch.float64, device=DEV),
               torch.zeros(H, dtype=torch.float64, device=DEV)) for s in slots}
    for prefixes in ([0] * len(lens), lens):                     # the second launch goes on from what the first one left
        a = torch.randn(T, 2 * H * (D + Dv), generator=g, device=DEV).bfloat16()          # views of one product
        q, k, v, gate = a.split([H * D, H * D, H * Dv, H * Dv], 1)
        ip, fp = torch.randn(T, H, generator=g, device=DEV) * 2, torch.randn(T, H, generator=g, device=DEV) * 2 + 1
        out = _native.mlstm_scan(q, k, v, gate, ip, fp, nw, S, n, m, seq_extend(lens, prefixes, slots), H, D, Dv, cap, eps)
        ig, fg = cap * torch.tanh(ip.double() / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(fp.double() / cap))
        want, at = torch.empty(T, H, Dv, dtype=torch.float64, device=DEV), 0
        for length, slot in zip(lens, slots):
            Sr, nr, mr = ref[slot]
            for t in range(at, at + length):
                qt, kt, vt = q[t].double().view(H, D) * D ** -0.5, k[t].double().view(H, D), v[t].double().view(H, Dv)
                top = torch.maximum(fg[t] + mr, ig[t])
                keep, take = torch.exp(fg[t] + mr - top), torch.exp(ig[t] - top)
                mr = top
                Sr = keep[:, None, None] * Sr + take[:, None, None] * kt[:, :, None] * vt[:, None]
                nr = keep[:, None] * nr + take[:, None] * kt
                den = torch.maximum((nr * qt).sum(-1).abs(), torch.exp(-mr)) + 1e-6
                want[t] = (Sr * qt[:, :, None]).sum(1) / den[:, None]
            ref[slot] = (Sr, nr, mr)
            at += length
            near(S[slot], Sr, 2e-5)
            near(n[slot], nr, 2e-5)
            assert (m[slot].double() - mr).abs().max() <= 2e-5 * max(1.0, mr.abs().max())
        want = want / torch.sqrt((want * want).mean(-1, keepdim=True) + eps)
        want = want.view(T, H * Dv) * nw.double() * torch.sigmoid(gate.double())
        # bf16 result: half an ulp (2^-9) of it, and what near-cancelling normalisers amplify of the fp32 sums
        assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-3).all()
    for slot in range(0, n_slots, 2):                            # no other slot was touched
        assert torch.isnan(S[slot]).all() and torch.isnan(n[slot]).all() and torch.isnan(m[slot]).all()


@pytest.mark.parametrize("lens", LENS, ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,G,N,Dv", [(4, 2, 128, 64), (2, 1, 128, 128), (3, 3, 64, 128), (6, 2, 64, 64)])
def test_mamba2_chunks(lens, H, G, N, Dv):
    from scratchpad_amd import _native
    announce("mamba2 chunks", lens, H, G, N, Dv)
    g = torch.Generator(device=DEV).manual_seed(4)
    T, slots = sum(lens), slots_of(lens)
    n_slots = 2 * len(lens) + 1
    S = torch.full((n_slots, H, N, Dv), float("nan"), device=DEV)
    A, bias, skip = (torch.randn(H, generator=g, device=DEV) * 0.5 - 1 for _ in range(3))
    ref = {s: torch.zeros(H, N, Dv, dtype=torch.float64, device=DEV) for s in slots}
    for prefixes in ([0] * len(lens), lens):
        xbc = torch.randn(T, H * Dv + 2 * G * N, generator=g, device=DEV).bfloat16()
        raw = torch.randn(T, H, generator=g, device=DEV)
        y = _native.mamba2_scan(xbc, raw, bias, A, skip, S, seq_extend(lens, prefixes, slots), H, G, N, Dv)
        x = xbc[:, :H * Dv].double().view(T, H, Dv)
        B, C = (xbc[:, H * Dv + i * G * N:H * Dv + (i + 1) * G * N].double().view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
        dt = torch.nn.functional.softplus(raw.double() + bias.double())
        dec = torch.exp(-torch.exp(A.double()) * dt)
        want, at = torch.empty(T, H, Dv, dtype=torch.float64, device=DEV), 0
        for length, slot in zip(lens, slots):
            Sr = ref[slot]
            for t in range(at, at + length):
                Sr = dec[t][:, None, None] * Sr + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None]
                want[t] = (Sr * C[t][:, :, None]).sum(1) + skip.double()[:, None] * x[t]
            ref[slot] = Sr
            at += length
            near(S[slot], Sr, 2e-5)
        near(y.view(T, H, Dv), want, 2e-5)
    for slot in range(0, n_slots, 2):
        assert torch.isnan(S[slot]).all()


DELTA_LENS = [[8], [15, 16, 17], [48, 1, 33, 2], [16, 200, 3]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", DELTA_LENS, ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,G,D,Dv", [(2, 1, 128, 128), (4, 4, 64, 64), (3, 3, 128, 48), (2, 2, 64, 208)])
def test_gated_delta_chunks(lens, H, G, D, Dv, dtype):
    from scratchpad_amd import _native
    announce("gated delta chunks", dtype, lens, H, G, D, Dv)
    g = torch.Generator(device=DEV).manual_seed(5)
    T, slots = sum(lens), slots_of(lens)
    n_slots = 2 * len(lens) + 1
    S = torch.full((n_slots, H, D, Dv), float("nan"), device=DEV)
    ref = {s: torch.zeros(H, D, Dv, dtype=torch.float64, device=DEV) for s in slots}
    nw = torch.rand(Dv, generator=g, device=DEV) + 0.5
    for prefixes in ([0] * len(lens), lens):
        a = torch.randn(T, 2 * G * D + H * Dv + H, generator=g, device=DEV).to(dtype)
        q, k, v, bp = a.split([G * D, G * D, H * Dv, H], 1)
        if not _native._delta_chunks_take(q, k, v, None, seq_extend(lens, prefixes, slots), D, Dv):
            q, k = q.contiguous(), k.contiguous()                # (a product whose width breaks the rows' alignment)
        decay = torch.rand(T, H * D, generator=g, device=DEV) ** 2
        decay[torch.rand(T, H * D, generator=g, device=DEV) < 0.05] = 0.0          # a channel forgotten, and one kept, exactly
        decay[:, 0] = 1.0
        gate = torch.rand(T, H * Dv, generator=g, device=DEV)
        seq = seq_extend(lens, prefixes, slots)
        assert _native._delta_chunks_take(q, k, v, decay, seq, D, Dv)
        out = _native.gated_delta_scan(q, k, v, bp, decay, gate, nw, S, seq, H, G, D, Dv, 1e-5)
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        kk, qq = (unit(x.double().view(T, G, D)).repeat_interleave(H // G, 1) for x in (k, q))
        qq, vv, beta = qq * D ** -0.5, v.double().view(T, H, Dv), torch.sigmoid(bp.double())
        w, want, at = decay.double().view(T, H, D), torch.empty(T, H, Dv, dtype=torch.float64, device=DEV), 0
        for length, slot in zip(lens, slots):
            Sr = ref[slot]
            for t in range(at, at + length):
                Sr = w[t][:, :, None] * Sr
                u = beta[t][:, None] * (vv[t] - (Sr * kk[t][:, :, None]).sum(1))
                Sr = Sr + kk[t][:, :, None] * u[:, None]
                want[t] = (Sr * qq[t][:, :, None]).sum(1)
            ref[slot] = Sr
            at += length
            near(S[slot], Sr, 2e-5)
        want = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5)
        want = (want * nw.double()).view(T, H * Dv) * gate.double()
        bar = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10, torch.float32: 1e-4}[dtype]
        # (1e-3: a head whose read-out nearly cancels is scaled up by its norm, and the fp32 sums' roundings with it)
        assert ((out.double() - want).abs() <= bar * want.abs() + 1e-3).all()
    for slot in range(0, n_slots, 2):
        assert torch.isnan(S[slot]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", DELTA_LENS, ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,G,D,Dv", [(2, 1, 128, 128), (4, 4, 64, 64), (3, 3, 128, 48), (2, 2, 64, 208)])
def test_gated_delta_chunks_where_the_other_form_pays(lens, H, G, D, Dv, dtype, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    test_gated_delta_chunks(lens, H, G, D, Dv, dtype)


def test_gated_delta_chunks_of_any_decays():
    """products of up to 16 decays are formed and never quotients: zeros, negative ones and ones above 1 are numbers like others"""
    from scratchpad_amd import _native
    announce("gated delta chunks of any decays")
    g = torch.Generator(device=DEV).manual_seed(7)
    lens, slots, H, D, Dv = [48, 33], [1, 3], 2, 64, 64
    T, seq = sum(lens), seq_extend([48, 33], [0, 0], [1, 3])
    q, k, v, bp = (torch.randn(T, n, generator=g, device=DEV) for n in (H * D, H * D, H * Dv, H))
    decay = torch.rand(T, H * D, generator=g, device=DEV) * 2.1 - 1.05
    decay[::5] = 0.0
    S, gate, nw = torch.zeros(4, H, D, Dv, device=DEV), torch.ones(T, H * Dv, device=DEV), torch.ones(Dv, device=DEV)
    assert _native._delta_chunks_take(q, k, v, decay, seq, D, Dv)
    _native.gated_delta_scan(q, k, v, bp, decay, gate, nw, S, seq, H, H, D, Dv, 1e-5)
    kk = k.double().view(T, H, D)
    kk, beta, w = kk / torch.sqrt((kk * kk).sum(-1, keepdim=True) + 1e-6), torch.sigmoid(bp.double()), decay.double().view(T, H, D)
    at = 0
    for length, slot in zip(lens, slots):
        Sr = torch.zeros(H, D, Dv, dtype=torch.float64, device=DEV)
        for t in range(at, at + length):
            Sr = w[t][:, :, None] * Sr
            u = beta[t][:, None] * (v[t].double().view(H, Dv) - (Sr * kk[t][:, :, None]).sum(1))
            Sr = Sr + kk[t][:, :, None] * u[:, None]
        at += length
        near(S[slot], Sr, 2e-5)


@pytest.mark.parametrize("T", [64, 129, 700])
@pytest.mark.parametrize("rank,channels", [(32, 16), (64, 208), (96, 64), (128, 2048)])
def test_lowrank_gate_of_many_tokens(T, rank, channels):
    from scratchpad_amd import _native
    announce("lowrank_gate", T, rank, channels)
    g = torch.Generator(device=DEV).manual_seed(6)
    p = torch.randn(T, rank + 8, generator=g, device=DEV).bfloat16()[:, 8:]
    w2t, bias = torch.randn(rank, channels, generator=g, device=DEV) * rank ** -0.5, torch.randn(channels, generator=g, device=DEV)
    A = torch.randn(channels // 16, generator=g, device=DEV) * 0.5 - 1
    z = p.double() @ w2t.double() + bias.double()
    want = torch.exp(-torch.exp(A.double()).repeat_interleave(16) * torch.nn.functional.softplus(z))
    # a decay moves by its exponent's error: fp32 sums of `rank` products, a few ulp of exponential and logarithm
    assert ((_native.lowrank_gate(p, w2t, bias, "decay", A).double() - want).abs() <= 4e-6).all()
    assert ((_native.lowrank_gate(p, w2t, None, "sigmoid").double() - torch.sigmoid(p.double() @ w2t.double())).abs() <= 2e-6).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", [[18], [15, 32, 17], [48, 1, 33, 2], [16, 200, 3]], ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,G,D,Dv", [(2, 1, 128, 128), (4, 4, 64, 64), (3, 3, 128, 48), (2, 2, 64, 256)])
def test_head_delta_chunks_against_the_per_token_kernel(lens, H, G, D, Dv, dtype):
    """Both orders of the same fp32 sums: S within 2e-5 of its largest value, as the channel-gated form is held to, and the normed
    read-outs within two roundings of the result"""
    from scratchpad_amd import _native
    announce("head delta chunks", dtype, lens, H, G, D, Dv)
    g = torch.Generator(device=DEV).manual_seed(6)
    T, slots = sum(lens), slots_of(lens)
    S = torch.full((2 * len(lens) + 1, H, D, Dv), float("nan"), device=DEV)
    S2 = S.clone()
    nw, dt_bias, A_log = (torch.rand(n, generator=g, device=DEV) for n in (Dv, H, H))
    for prefixes in ([0] * len(lens), lens):
        q, k, v, gate = (torch.randn(T, n, generator=g, device=DEV).to(dtype) for n in (G * D, G * D, H * Dv, H * Dv))
        pre = torch.randn(T, 2 * H, generator=g, device=DEV)
        pre[T // 2, H:] = 60.0                                                     # a head forgotten all but exactly
        seq = seq_extend(lens, prefixes, slots)
        assert _native._delta_chunks_take(q, k, v, None, seq, D, Dv) == (T >= 18 * len(lens))
        if T < 18 * len(lens):
            return
        args = (q, k, v, gate, pre, dt_bias, A_log, nw)
        out = _native.head_delta_scan(*args, S, seq, H, G, D, Dv, 1e-5)
        want = _native.head_delta_scan(*args, S2, seq, H, G, D, Dv, 1e-5, ranges=1)
        for slot in slots:
            near(S[slot], S2[slot].double(), 2e-5)
        bar = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -9, torch.float32: 1e-4}[dtype]
        assert ((out.double() - want.double()).abs() <= bar * want.double().abs() + 1e-3).all()
    for slot in range(0, 2 * len(lens) + 1, 2):
        assert torch.isnan(S[slot]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", [[18], [15, 32, 17], [16, 200, 3]], ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,G,D,Dv", [(2, 1, 128, 128), (4, 4, 64, 64), (3, 3, 128, 48), (2, 2, 64, 256)])
def test_head_delta_chunks_where_the_other_form_pays(lens, H, G, D, Dv, dtype, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    test_head_delta_chunks_against_the_per_token_kernel(lens, H, G, D, Dv, dtype)


MANY = [17, 5, 33, 16] * 24      # 288 workgroups of 3 heads: the widest range of columns per workgroup


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
def test_delta_chunks_of_many_requests(D, dtype, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    test_gated_delta_chunks(MANY, 3, 1, D, 128, dtype)
    test_head_delta_chunks_against_the_per_token_kernel([n + 16 for n in MANY], 3, 1, D, 128, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,Dv", [(128, 128), (64, 48)])
def test_gated_delta_chunks_of_rows_of_any_length(D, Dv, dtype, monkeypatch):
    """q and k are of unit length whatever they come as: the chunks' products of rows of 1e-6 to 1e6 against the per-token kernel's, both
    orders of the same fp32 sums (bars as above)"""
    from scratchpad_amd import _native
    announce("gated delta rows of any length", dtype, D, Dv)
    g = torch.Generator(device=DEV).manual_seed(9)
    lens, H = [50, 17, 32], 2
    T, slots = sum(lens), slots_of(lens)
    size = lambda: 10.0 ** (12 * torch.rand(T, 1, generator=g, device=DEV) - 6)  # noqa: E731
    q, k = ((torch.randn(T, H * D, generator=g, device=DEV) * size()).to(dtype) for _ in range(2))
    v, bp = (torch.randn(T, n, generator=g, device=DEV).to(dtype) for n in (H * Dv, H))
    decay, gate = (torch.rand(T, n, generator=g, device=DEV) for n in (H * D, H * Dv))
    nw, states, outs = torch.rand(Dv, generator=g, device=DEV) + 0.5, [], []
    for chunks in (True, False):
        monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a, chunks=chunks: chunks)
        states.append(torch.zeros(2 * len(lens) + 1, H, D, Dv, device=DEV))
        outs.append(_native.gated_delta_scan(q, k, v, bp, decay, gate, nw, states[-1], seq_extend(lens, [0] * len(lens), slots), H, H, D, Dv, 1e-5))
    for slot in slots:
        near(states[0][slot], states[1][slot].double(), 2e-5)
    bar = {torch.bfloat16: 2.0 ** -7, torch.float32: 1e-4}[dtype]
    # (1e-3: as in test_gated_delta_chunks)
    assert ((outs[0].double() - outs[1].double()).abs() <= bar * outs[1].double().abs() + 1e-3).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("channel", [True, False], ids=["gated", "head"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows,values", [(1e18, 1e21), (0.0, 1e36)])
def test_delta_chunks_of_states_at_the_end_of_fp32(rows, values, D, channel, dtype, monkeypatch):
    """q and k enter every product with unit length: long rows beside large states, and rows of zeros beside the largest values, leave the states
    that the per-token kernels leave, two orders of the same fp32 sums (bar as above)"""
    from scratchpad_amd import _native
    announce("delta states at the end of fp32", dtype, D, channel, rows, values)
    g = torch.Generator(device=DEV).manual_seed(21)
    lens, H, Dv = [50, 17, 32], 2, 128
    T, slots = sum(lens), slots_of(lens)
    size = torch.where(torch.arange(T, device=DEV) % 3 == 1, rows, 1.0)[:, None]
    q, k = ((torch.randn(T, H * D, generator=g, device=DEV) * size).to(dtype) for _ in range(2))
    v, bp = (torch.randn(T, H * Dv, generator=g, device=DEV) * values).to(dtype), torch.randn(T, H, generator=g, device=DEV).to(dtype)
    decay, gate, pre = (torch.rand(T, n, generator=g, device=DEV) for n in (H * D, H * Dv, 2 * H))
    nw, dt_bias, A_log, states = torch.ones(Dv, device=DEV), *(torch.rand(H, generator=g, device=DEV) for _ in range(2)), []
    seq = seq_extend(lens, [0] * len(lens), slots)
    for chunks in (True, False):
        monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a, chunks=chunks: chunks)
        S = torch.zeros(2 * len(lens) + 1, H, D, Dv, device=DEV)
        if channel:
            _native.gated_delta_scan(q, k, v, bp, decay, gate, nw, S, seq, H, H, D, Dv, 1e-5)
        else:
            _native.head_delta_scan(q, k, v, gate.to(dtype), pre, dt_bias, A_log, nw, S, seq, H, H, D, Dv, 1e-5)
        states.append(S)
    for slot in slots:
        near(states[0][slot], states[1][slot].double(), 2e-5)


def _unit_parts_just_below_a_cut(lo, factor, n, seed):
    """n pairs (a, b) of fp32 whose unit row's a, times `factor`, lies in [lo, 1.06 lo] with mantissas that split badly into 8 + 8 + 8 bits:
    below a cut of the first, half of one of the second left over"""
    g, out = torch.Generator().manual_seed(seed), []
    while len(out) < n:
        a = lo / factor * (1 + 0.06 * torch.rand(1 << 20, generator=g))
        b = torch.sqrt(1 - a * a)
        x = a * (factor / torch.sqrt(a * a + b * b + 1e-6))
        low = x.view(torch.int32) & 0xffff
        hit = ((low >= 0xff60) & (low <= 0xff7e)).nonzero()[:, 0]
        out += [(float(a[i]), float(b[i])) for i in hit]
    return torch.tensor(out[:n])


@pytest.mark.parametrize("D", [64, 128])
def test_delta_products_of_one_channel_are_products_in_fp32(D, monkeypatch):
    """Sums that one channel makes up: a product k v of the state and a product q S of the read-out, of mantissas whose parts of 8 bits leave the
    most behind.  fp32 rounds the product (at most 2^-24 of it, 2^-24 / sqrt(3) in the mean), the read-out's norm once more for each of two columns."""
    from scratchpad_amd import _native
    announce("delta products of one channel", D)
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    H, Dv, T, ulp = 2, 64, 16, 2.0 ** -24
    g = torch.Generator().manual_seed(7)
    # columns: 1, then numbers just below a cut over some exponents and signs
    low = 0xff60 + torch.randint(0, 0x1f, (T, Dv), generator=g)
    bits = (torch.randint(125, 130, (T, Dv), generator=g) << 23) | (torch.randint(0, 8, (T, Dv), generator=g) << 16) | low
    numbers = bits.int().view(torch.float32) * (1 - 2 * torch.randint(0, 2, (T, Dv), generator=g))
    numbers[:, 0] = 1.0
    seq = lambda held: seq_extend([T], [held], [1])  # noqa: E731
    ones = lambda n: torch.ones(T, n, device=DEV)  # noqa: E731
    rows = lambda pairs: torch.stack([torch.nn.functional.pad(p, (2 * t, D - 2 * t - 2)) for t, p in enumerate(pairs)]).repeat(1, H).to(DEV)  # noqa: E731

    def error(got, want):
        return float(((got / want - 1) ** 2).mean().sqrt() / ulp)

    # S = k v: token t has the channels 2 t and 2 t + 1 to itself, steps of 1, no decay; the column of ones is k
    S = torch.zeros(2, H, D, Dv, device=DEV)
    k = rows(_unit_parts_just_below_a_cut(0.5, 1.0, T, 1))
    v = numbers.repeat(1, H).to(DEV)
    _native.gated_delta_scan(k, k, v, ones(H) * 100, ones(H * D), ones(H * Dv), torch.ones(Dv, device=DEV), S, seq(0), H, H, D, Dv, 1e-5)
    got = S[1, :, 0:2 * T:2].double().cpu()                                       # [H, T, Dv]
    assert error(got[:, :, 1:], got[:, :, :1] * numbers[:, 1:].double()) <= 1.0

    # o = q S of a held state whose rows 2 t are the numbers and rows 2 t + 1 zeros; keys of zeros leave it
    S = torch.zeros(2, H, D, Dv, device=DEV)
    S[1, :, 0:2 * T:2] = numbers.to(DEV)
    q = rows(_unit_parts_just_below_a_cut(2.0 ** -4, D ** -0.5, T, 2))
    out = _native.gated_delta_scan(q, torch.zeros_like(q), torch.zeros_like(v), ones(H), ones(H * D), ones(H * Dv), torch.ones(Dv, device=DEV), S, seq(16),
                                   H, H, D, Dv, 1e-5)
    got = out.view(T, H, Dv).double().cpu()
    assert error(got[:, :, 1:], got[:, :, :1] * numbers[:, None, 1:].double()) <= 1.5


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.bfloat16, 32), (torch.float32, 64)])
@pytest.mark.parametrize("lens", [[1, 1, 1], [70, 3]], ids=lambda l: "-".join(map(str, l)))
def test_mlstm_gates_as_halves_of_one_product(dtype, D, lens):
    """the bits of the scan on contiguous gates, in prompts and (one token each) in steps, for the chunk and the per-token kernels"""
    from scratchpad_amd import _native
    announce("mlstm gates", dtype, D, lens)
    g = torch.Generator(device=DEV).manual_seed(9)
    T, H, slots = sum(lens), 2, slots_of(lens)
    q, k, v, gate = (torch.randn(T, H * D, generator=g, device=DEV).to(dtype) for _ in range(4))
    gates, nw = torch.randn(T, 2 * H, generator=g, device=DEV), torch.rand(H * D, generator=g, device=DEV)
    ip, fp = gates[:, :H], gates[:, H:]
    got = []
    for i, f in ((ip, fp), (ip.contiguous(), fp.contiguous()), (ip, fp.contiguous())):
        S, n, m = (torch.zeros(2 * len(lens) + 1, H, *w, device=DEV) for w in ((D, D), (D,), ()))
        seq = _native.SeqParams(torch.tensor(slots, device=DEV), torch.tensor([5] * len(lens), device=DEV)) if max(lens) == 1 \
            else seq_extend(lens, [0] * len(lens), slots)
        got.append((_native.mlstm_scan(q, k, v, gate, i, f, nw, S, n, m, seq, H, D, D, 15.0, 1e-5), S, n, m))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))


def mamba2_in_64_bits(xbc, raw, bias, A, skip, lens, H, G, N, Dv):
    """(outputs [T, H, Dv], the requests' states) from empty states"""
    T = xbc.shape[0]
    x = xbc[:, :H * Dv].double().view(T, H, Dv)
    B, C = (xbc[:, H * Dv + i * G * N:H * Dv + (i + 1) * G * N].double().view(T, G, N).repeat_interleave(H // G, 1) for i in (0, 1))
    dt = torch.nn.functional.softplus(raw.double() + bias.double())
    dec = torch.exp(-torch.exp(A.double()) * dt)
    want, at, states = torch.empty(T, H, Dv, dtype=torch.float64, device=DEV), 0, []
    for length in lens:
        S = torch.zeros(H, N, Dv, dtype=torch.float64, device=DEV)
        for t in range(at, at + length):
            S = dec[t][:, None, None] * S + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None]
            want[t] = (S * C[t][:, :, None]).sum(1) + skip.double()[:, None] * x[t]
        states.append(S)
        at += length
    return want, states


@pytest.mark.parametrize("kind", ["rates to 16", "large steps before small ones", "forgotten at once"])
def test_mamba2_chunks_of_strong_decays(kind):
    """The weight of one token at another is the exponential of a difference of summed log decays, which reach -1000 and more in a
    chunk: were the sums rounded to fp32 before they are subtracted, weights would be off by up to 6e-5.  What fp32 gives is an ulp of
    the difference itself (below 10 where a weight matters), of the rate and of the sums: 4e-6 of a head's largest value."""
    from scratchpad_amd import _native
    announce("mamba2 strong decays", kind)
    g = torch.Generator(device=DEV).manual_seed(14)
    lens, H, G, N, Dv = [200, 65], 4, 1, 64, 64
    T, slots = sum(lens), [1, 3]
    A = torch.log(torch.tensor([1.0, 4.0, 16.0, 16.0], device=DEV))
    raw, bias = torch.randn(T, H, generator=g, device=DEV), torch.zeros(H, device=DEV)
    if kind.startswith("large"):
        raw.fill_(-5.0)                                              # steps of 0.0067 ...
        raw[::64], raw[20::64] = 50.0, 30.0                          # ... between steps of 50 and 30
    if kind.startswith("forgotten"):
        A[2] = 95.0                                                  # e^95 is past fp32: every decay is zero
    xbc, skip = torch.randn(T, H * Dv + 2 * G * N, generator=g, device=DEV).bfloat16(), torch.zeros(H, device=DEV)
    S = torch.full((5, H, N, Dv), float("nan"), device=DEV)
    y = _native.mamba2_scan(xbc, raw, bias, A, skip, S, seq_extend(lens, [0, 0], slots), H, G, N, Dv).view(T, H, Dv)
    want, states = mamba2_in_64_bits(xbc, raw, bias, A, skip, lens, H, G, N, Dv)
    for h in range(H):
        near(y[:, h], want[:, h], 4e-6)
        for slot, ref in zip(slots, states):
            near(S[slot, h], ref[h], 4e-6)


@pytest.mark.parametrize("length", [1, 10, 11])
def test_mamba2_short_portions_of_many_requests(length):
    """on both sides of the line between the forms, and with the number of rows not given: the same numbers within fp32's sums"""
    from scratchpad_amd import _native
    announce("mamba2 short portions", length)
    g = torch.Generator(device=DEV).manual_seed(19)
    B, H, G, N, Dv = 64, 32, 1, 64, 64
    T, slots = B * length, list(range(1, B + 1))
    xbc, raw = torch.randn(T, H * Dv + 2 * G * N, generator=g, device=DEV).bfloat16(), torch.randn(T, H, generator=g, device=DEV)
    A, bias, skip = (torch.randn(H, generator=g, device=DEV) * 0.5 - 1 for _ in range(3))
    seq = seq_extend([length] * B, [0] * B, slots)
    want, states = mamba2_in_64_bits(xbc, raw, bias, A, skip, [length] * B, H, G, N, Dv)
    S = torch.zeros(2, B + 1, H, N, Dv, device=DEV)
    y = [_native.mamba2_scan(xbc, raw, bias, A, skip, S[0], seq, H, G, N, Dv), torch.empty(T, H * Dv, device=DEV)]
    _native._check(_native.load().sp_mamba2_scan(y[1].data_ptr(), H * Dv, xbc.data_ptr(), xbc.stride(0), raw.data_ptr(), bias.data_ptr(),
                                                 A.data_ptr(), skip.data_ptr(), S[1].data_ptr(), S[1].stride(0), H, G, N, Dv, *seq.args,
                                                 _native._dt(xbc), _native._stream()), "sp_mamba2_scan")
    for i in (0, 1):
        near(y[i].view(T, H, Dv), want, 2e-6)
        near(S[i][1:], torch.stack(states), 2e-6)


@pytest.mark.parametrize("length", [1, 6, 7])
def test_mlstm_short_portions_of_many_requests(length):
    """the same numbers within fp32's sums on both sides of the line between the forms (6 tokens), with the number of rows given and not"""
    from scratchpad_amd import _native
    announce("mlstm short portions", length)
    g = torch.Generator(device=DEV).manual_seed(20)
    B, H, D = 64, 16, 64
    T, slots = B * length, list(range(1, B + 1))
    q, k, v, gate = (torch.randn(T, H * D, generator=g, device=DEV).bfloat16() for _ in range(4))
    ip, fp, nw = torch.randn(T, H, generator=g, device=DEV), torch.randn(T, H, generator=g, device=DEV) + 1, torch.ones(H * D, device=DEV)
    seq, got = seq_extend([length] * B, [0] * B, slots), []
    for known in (True, False):
        S, n, m = torch.zeros(B + 1, H, D, D, device=DEV), torch.zeros(B + 1, H, D, device=DEV), torch.zeros(B + 1, H, device=DEV)
        if known:
            y = _native.mlstm_scan(q, k, v, gate, ip, fp, nw, S, n, m, seq, H, D, D, 15.0, 1e-5)
        else:
            y = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
            _native._check(_native.load().sp_mlstm_scan(
                y.data_ptr(), H * D, q.data_ptr(), H * D, k.data_ptr(), H * D, v.data_ptr(), H * D, gate.data_ptr(), H * D, ip.data_ptr(),
                fp.data_ptr(), nw.data_ptr(), S.data_ptr(), S.stride(0), n.data_ptr(), n.stride(0), m.data_ptr(), m.stride(0), H, D, D,
                15.0, 1e-5, *seq.args, _native._dt(q), _native._stream()), "sp_mlstm_scan")
        got.append((y, S, n, m))
    (y0, *a), (y1, *b) = got
    for x, w in zip(a, b):
        near(x, w.double(), 2e-6)
    # two roundings of a result of 8 bits; a normaliser that nearly cancels scales fp32's sums up
    assert ((y0.double() - y1.double()).abs() <= 2.0 ** -7 * y1.double().abs() + 2e-3).all()


def test_mlstm_chunks_of_closed_forget_gates():
    """A chunk whose first 16 tokens forget nothing and whose others forget all but e^-15 each: the summed log gates reach -700, and a
    weight taken from sums rounded to fp32 would be off by 3e-5.  Half of the values cancel in pairs (k is the same everywhere, v
    alternates), so that what is left of them is 1e-3 of a weight; the other half is of that size and adds up.  Their ratio is what the
    norm keeps: an error of 3e-5 would be percents of it, fp32's 1e-7 is below the result's 16-bit rounding."""
    from scratchpad_amd import _native
    announce("mlstm closed gates")
    H, D, T = 2, 64, 64
    g = torch.Generator(device=DEV).manual_seed(15)
    one = torch.randn(1, H * D, generator=g, device=DEV).bfloat16()
    k = q = one.expand(T, H * D).contiguous()
    v = torch.ones(T, H * D, device=DEV)
    v[1::2] = -1.0
    v[:, 1::2] = 1e-4
    v, gate = v.bfloat16(), torch.full((T, H * D), 3.0, device=DEV).bfloat16()
    ip = torch.full((T, H), 0.25, device=DEV)
    fp = torch.full((T, H), -40.0, device=DEV)
    fp[:16] = 10.0
    nw, cap, eps = torch.ones(H * D, device=DEV), 15.0, 1e-14
    S, n, m = torch.zeros(2, H, D, D, device=DEV), torch.zeros(2, H, D, device=DEV), torch.zeros(2, H, device=DEV)
    out = _native.mlstm_scan(q, k, v, gate, ip, fp, nw, S, n, m, seq_extend([T], [0], [1]), H, D, D, cap, eps)
    ig, fg = cap * torch.tanh(ip.double() / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(fp.double() / cap))
    Sr, nr, mr = (torch.zeros(H, *w, dtype=torch.float64, device=DEV) for w in ((D, D), (D,), ()))
    for t in range(16):
        qt, kt, vt = q[t].double().view(H, D) * D ** -0.5, k[t].double().view(H, D), v[t].double().view(H, D)
        top = torch.maximum(fg[t] + mr, ig[t])
        keep, take = torch.exp(fg[t] + mr - top), torch.exp(ig[t] - top)
        mr = top
        Sr = keep[:, None, None] * Sr + take[:, None, None] * kt[:, :, None] * vt[:, None]
        nr = keep[:, None] * nr + take[:, None] * kt
        o = (Sr * qt[:, :, None]).sum(1) / (torch.maximum((nr * qt).sum(-1).abs(), torch.exp(-mr)) + 1e-6)[:, None]
        want = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * torch.sigmoid(gate[t].double()).view(H, D)
        if t % 2:                                                    # (the pairs are whole)
            assert ((out[t].double().view(H, D) - want).abs() <= 2.0 ** -8 * want.abs() + 2e-3).all(), t


BAD = [float("nan"), float("inf"), float("-inf")]


@pytest.mark.parametrize("bad", BAD, ids=str)
@pytest.mark.parametrize("at", [0, 5, 40, 63, 70, 129])
def test_mamba2_values_that_are_not_finite_reach_no_earlier_token(bad, at):
    """... and no other column, head or request: all of that keeps the bits of a launch without them"""
    from scratchpad_amd import _native
    announce("mamba2 not finite", bad, at)
    g = torch.Generator(device=DEV).manual_seed(16)
    lens, H, G, N, Dv = [130, 20], 2, 1, 64, 64
    T, slots = sum(lens), [1, 3]
    A, bias, skip = (torch.randn(H, generator=g, device=DEV) * 0.5 - 1 for _ in range(3))
    raw = torch.randn(T, H, generator=g, device=DEV)
    clean = torch.randn(T, H * Dv + 2 * G * N, generator=g, device=DEV).bfloat16()
    dirty = clean.clone()
    dirty[at, Dv + 7] = bad                                          # head 1, column 7
    got = []
    for xbc in (clean, dirty):
        S = torch.zeros(5, H, N, Dv, device=DEV)
        got.append((_native.mamba2_scan(xbc, raw, bias, A, skip, S, seq_extend(lens, [0, 0], slots), H, G, N, Dv).view(T, H, Dv), S))
    (y0, S0), (y1, S1) = got
    hit = torch.zeros(T, H, Dv, dtype=torch.bool, device=DEV)
    hit[at:130, 1, 7] = True
    assert torch.equal(y1[~hit], y0[~hit]) and not torch.isfinite(y1[hit]).any()
    hit = torch.zeros_like(S0, dtype=torch.bool)
    hit[1, 1, :, 7] = True
    assert torch.equal(S1[~hit], S0[~hit]) and not torch.isfinite(S1[hit]).any()


# (an infinite gate is capped)
@pytest.mark.parametrize("where,bad", [(w, b) for w in "qkv" for b in BAD] + [("ipre", BAD[0]), ("fpre", BAD[0])])
@pytest.mark.parametrize("at", [0, 40, 63, 70])
def test_mlstm_values_that_are_not_finite_reach_no_earlier_token(at, where, bad):
    from scratchpad_amd import _native
    announce("mlstm not finite", where, bad, at)
    g = torch.Generator(device=DEV).manual_seed(17)
    lens, H, D = [100, 20], 2, 64
    T, slots = sum(lens), [1, 3]
    clean = {x: torch.randn(T, H * D, generator=g, device=DEV).bfloat16() for x in ("q", "k", "v", "gate")}
    clean.update({x: torch.randn(T, H, generator=g, device=DEV) + 1 for x in ("ipre", "fpre")})
    dirty = {x: t.clone() for x, t in clean.items()}
    dirty[where][at, 1 if where[1:] == "pre" else D + 7] = bad       # head 1
    nw, got = torch.rand(H * D, generator=g, device=DEV) + 0.5, []
    for x in (clean, dirty):
        S, n, m = torch.zeros(5, H, D, D, device=DEV), torch.zeros(5, H, D, device=DEV), torch.zeros(5, H, device=DEV)
        got.append((_native.mlstm_scan(x["q"], x["k"], x["v"], x["gate"], x["ipre"], x["fpre"], nw, S, n, m,
                                       seq_extend(lens, [0, 0], slots), H, D, D, 15.0, 1e-5).view(T, H, D), S, n))
    (y0, S0, n0), (y1, S1, n1) = got
    hit = torch.zeros(T, H, D, dtype=torch.bool, device=DEV)
    hit[at:at + 1 if where == "q" else 100, 1] = True                # a query touches its own token only
    assert torch.equal(y1[~hit], y0[~hit]) and not torch.isfinite(y1[hit]).any()
    assert torch.equal(S1[:, 0], S0[:, 0]) and torch.equal(S1[3], S0[3]) and torch.equal(n1[3], n0[3])
    if where == "v":
        assert torch.equal(n1, n0) and not torch.isfinite(S1[1, 1, :, 7]).any()
        hit = torch.arange(D, device=DEV) == 7
        assert torch.equal(S1[1, 1][:, ~hit], S0[1, 1][:, ~hit])


# (an infinite step size or decay is a number)
@pytest.mark.parametrize("where,bad", [(w, b) for w in "qkv" for b in BAD] + [("beta", BAD[0]), ("decay", BAD[0])])
@pytest.mark.parametrize("at", [0, 9, 15, 16, 40])
@pytest.mark.parametrize("channel", [True, False], ids=["gated", "head"])
def test_delta_values_that_are_not_finite_reach_no_earlier_token(channel, at, where, bad):
    from scratchpad_amd import _native
    announce("delta not finite", channel, where, bad, at)
    g = torch.Generator(device=DEV).manual_seed(18)
    lens, H, D, Dv = [61, 30], 2, 64, 64
    T, slots = sum(lens), [1, 3]
    rn = lambda n: torch.randn(T, n, generator=g, device=DEV)  # noqa: E731
    clean = {"q": rn(H * D).bfloat16(), "k": rn(H * D).bfloat16(), "v": rn(H * Dv).bfloat16(), "gate": rn(H * Dv).bfloat16(),
             "beta": rn(H).bfloat16(), "decay": torch.rand(T, H * D, generator=g, device=DEV), "pre": rn(2 * H)}
    dirty = {x: t.clone() for x, t in clean.items()}
    if not channel and where in ("beta", "decay"):
        dirty["pre"][at, 1 + (H if where == "decay" else 0)] = bad
    else:
        dirty[where][at, 1 if where == "beta" else D + 7] = bad
    nw, dt_bias, A_log = (torch.rand(n, generator=g, device=DEV) for n in (Dv, H, H))
    seq, got = seq_extend(lens, [0, 0], slots), []
    for x in (clean, dirty):
        S = torch.zeros(5, H, D, Dv, device=DEV)
        if channel:
            assert _native._delta_chunks_take(x["q"], x["k"], x["v"], x["decay"], seq, D, Dv)
            y = _native.gated_delta_scan(x["q"], x["k"], x["v"], x["beta"], x["decay"], x["gate"].float().abs(), nw, S, seq, H, H, D, Dv, 1e-5)
        else:
            assert _native._delta_chunks_take(x["q"], x["k"], x["v"], None, seq, D, Dv)
            y = _native.head_delta_scan(x["q"], x["k"], x["v"], x["gate"], x["pre"], dt_bias, A_log, nw, S, seq, H, H, D, Dv, 1e-5)
        got.append((y.view(T, H, Dv), S))
    (y0, S0), (y1, S1) = got
    hit = torch.zeros(T, H, Dv, dtype=torch.bool, device=DEV)
    hit[at:at + 1 if where == "q" else 61, 1] = True
    assert torch.equal(y1[~hit], y0[~hit]) and not torch.isfinite(y1[hit]).any()
    assert torch.equal(S1[:, 0], S0[:, 0]) and torch.equal(S1[3], S0[3])
    if where == "v":
        hit = torch.arange(Dv, device=DEV) == 7
        assert torch.equal(S1[1, 1][:, ~hit], S0[1, 1][:, ~hit]) and not torch.isfinite(S1[1, 1][:, hit]).any()


@pytest.mark.parametrize("where,bad", [(w, b) for w in "qkv" for b in BAD] + [("beta", BAD[0]), ("decay", BAD[0])])
@pytest.mark.parametrize("at", [0, 9, 15, 40])
@pytest.mark.parametrize("channel", [True, False], ids=["gated", "head"])
def test_delta_products_of_parts_and_values_that_are_not_finite(channel, at, where, bad, monkeypatch):
    """heads of 128: what is not finite reaches its own token's rows and the ones behind it, of its own head"""
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    announce("delta parts not finite", channel, where, bad, at)
    g = torch.Generator(device=DEV).manual_seed(19)
    lens, H, D, Dv = [61, 30], 2, 128, 128
    T = sum(lens)
    rn = lambda n: torch.randn(T, n, generator=g, device=DEV)  # noqa: E731
    x = {"q": rn(H * D).bfloat16(), "k": rn(H * D).bfloat16(), "v": rn(H * Dv).bfloat16(), "beta": rn(H).bfloat16(),
         "decay": torch.rand(T, H * D, generator=g, device=DEV), "pre": rn(2 * H)}
    gate, nw, dt_bias, A_log = rn(H * Dv).bfloat16(), *(torch.rand(n, generator=g, device=DEV) for n in (Dv, H, H))
    seq, got = seq_extend(lens, [0, 0], [1, 3]), []
    for dirty in (False, True):
        if dirty and not channel and where in ("beta", "decay"):
            x["pre"][at, 1 + (H if where == "decay" else 0)] = bad
        elif dirty:
            x[where][at, 1 if where == "beta" else D + 7] = bad
        S = torch.zeros(5, H, D, Dv, device=DEV)
        assert _native._delta_chunks_take(x["q"], x["k"], x["v"], x["decay"] if channel else None, seq, D, Dv)
        if channel:
            y = _native.gated_delta_scan(x["q"], x["k"], x["v"], x["beta"], x["decay"], gate.float().abs(), nw, S, seq, H, H, D, Dv, 1e-5)
        else:
            y = _native.head_delta_scan(x["q"], x["k"], x["v"], gate, x["pre"], dt_bias, A_log, nw, S, seq, H, H, D, Dv, 1e-5)
        got.append((y.view(T, H, Dv), S))
    (y0, S0), (y1, S1) = got
    hit = torch.zeros(T, H, Dv, dtype=torch.bool, device=DEV)
    hit[at:at + 1 if where == "q" else 61, 1] = True
    assert torch.equal(y1[~hit], y0[~hit]) and not torch.isfinite(y1[hit]).any()
    assert torch.equal(S1[:, 0], S0[:, 0]) and torch.equal(S1[3], S0[3])
    if where == "v":
        hit = torch.arange(Dv, device=DEV) == 7
        assert torch.equal(S1[1, 1][:, ~hit], S0[1, 1][:, ~hit]) and not torch.isfinite(S1[1, 1][:, hit]).any()


@pytest.mark.parametrize("T", [40, 64, 129])
def test_lowrank_decays_of_all_rates(T):
    """exp(-rate softplus(z)) at the accuracy of fp32 functions - the product's, an ulp or two of softplus, rate and exponential -
    whichever form a step takes: rates to 16, softplus from 2e-9 (a channel that hardly forgets) up"""
    from scratchpad_amd import _native
    announce("lowrank_gate of all rates", T)
    rank, channels = 32, 1024
    p, w2t = torch.zeros(T, rank, device=DEV).bfloat16(), torch.zeros(rank, channels, device=DEV)
    bias = torch.linspace(-20, 15, channels // 8, device=DEV).repeat(8).contiguous()                     # z exactly
    A = torch.log(torch.tensor([0.05, 0.4, 1.0, 2.0, 4.0, 8.0, 12.0, 16.0], device=DEV))
    x = torch.exp(A.double()).repeat_interleave(channels // 8) * torch.nn.functional.softplus(bias.double())
    want = torch.exp(-x)
    got = _native.lowrank_gate(p, w2t, bias, "decay", A).double()
    # half an ulp of the result and its exponential's ulp; three roundings of the exponent (rate, softplus, their product)
    bar = want * (1.5 * 2.0 ** -23 + 6 * 2.0 ** -24 * x) + 1e-38
    assert ((got - want).abs() <= bar).all(), float(((got - want).abs() / bar).max())
    sig = torch.sigmoid(bias.double())
    assert ((_native.lowrank_gate(p, w2t, bias, "sigmoid").double() - sig).abs() <= 4 * 2.0 ** -23 * sig).all()


def test_lowrank_gate_of_infinite_inputs():
    from scratchpad_amd import _native
    T, rank, channels = 64, 64, 32
    p, w2t = torch.ones(T, rank, device=DEV).bfloat16(), torch.full((rank, channels), 0.5, device=DEV)
    p[3, 5], p[9, 60], p[17, 2] = float("inf"), float("-inf"), float("nan")
    w2t[7, 31] = float("inf")
    decay, sig = _native.lowrank_gate(p, w2t, None, "decay", torch.zeros(2, device=DEV)), _native.lowrank_gate(p, w2t, None, "sigmoid")
    plain = p.float() @ w2t                                           # (no infinity meets a zero: the sums are infinite, not NaN)
    assert torch.isnan(decay[17]).all() and torch.isnan(sig[17]).all()
    keep = torch.arange(T, device=DEV) != 17
    assert torch.isinf(plain[3]).all() and (plain[9, :31] == float("-inf")).all() and torch.isnan(plain[9, 31])
    for got, ref in ((decay, torch.exp(-torch.nn.functional.softplus(plain))), (sig, torch.sigmoid(plain))):
        assert torch.equal(torch.isnan(got[keep]), torch.isnan(ref[keep]))
        assert torch.allclose(got[keep], ref[keep], rtol=1e-5, atol=1e-6, equal_nan=True)


SEGMENT_LENS = [[129], [64, 300, 1], [128, 127, 500, 2, 65], [257] + [3] * 66 + [192]]


@pytest.mark.parametrize("lens", SEGMENT_LENS, ids=lambda l: "-".join(map(str, l[:5])))
@pytest.mark.parametrize("H,D,Dv", [(3, 128, 128), (2, 128, 64), (2, 64, 128), (5, 64, 64)])
def test_scans_in_segments(lens, H, D, Dv, monkeypatch):
    """segments of 64 and 128 tokens around their edges, from an empty and from a held state, more requests than lanes: against the
    64-bit recurrences, as the whole requests above"""
    from scratchpad_amd import _native
    for segment in (64, 128):
        monkeypatch.setattr(_native, "SCAN_SEGMENT", segment)
        test_mlstm_chunks(lens, H, D, Dv)
        test_mamba2_chunks(lens, 2 * H, H, D, Dv)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_segments_keep_a_number_that_is_not_finite_from_earlier_tokens(bad, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "SCAN_SEGMENT", 64)
    H, D, T, at = 2, 64, 320, 100
    g = torch.Generator(device=DEV).manual_seed(5)
    a = torch.randn(T, 4 * H * D, generator=g, device=DEV).bfloat16()
    gates, ones = torch.randn(T, 2 * H, generator=g, device=DEV), torch.ones(H * D, device=DEV)
    xbc, dt, zeros = torch.randn(T, 3 * H * D, generator=g, device=DEV).bfloat16(), torch.randn(T, H, generator=g, device=DEV), torch.zeros(H, device=DEV)

    def run(where):
        b, x, gt, d = a.clone(), xbc.clone(), gates.clone(), dt.clone()
        if where == "value":
            b[at, 2 * H * D + 3] = bad
            x[at, 3] = bad
        elif where == "gate":
            gt[at] = d[at] = float("nan")
        S, n, m = (torch.zeros(2, H, *s, device=DEV) for s in ((D, D), (D,), ()))
        seq = seq_extend([T], [0], [1])
        out = _native.mlstm_scan(*b.split([H * D] * 4, 1), gt[:, :H], gt[:, H:], ones, S, n, m, seq, H, D, D, 15.0, 1e-5)
        S2 = torch.zeros(2, H, D, D, device=DEV)
        y = _native.mamba2_scan(x, d, zeros, zeros, zeros, S2, seq, H, H, D, D)
        return out, y, S[1], S2[1]
    clean = run("nowhere")
    for where in ("value", "gate"):
        out, y, S, S2 = run(where)
        assert torch.equal(out[:at], clean[0][:at]) and torch.equal(y[:at], clean[1][:at])
        cols = [3] if where == "value" else list(range(D))
        assert not torch.isfinite(S[0][:, cols]).any() and not torch.isfinite(S2[0][:, cols]).any()
        assert not torch.isfinite(out[at:].view(-1, H, D)[:, 0, cols].float()).any() and not torch.isfinite(y[at:].view(-1, H, D)[:, 0, cols]).any()


@pytest.mark.parametrize("lens", [[20], [9, 130, 300], [128], [17] * 3], ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("H,D,Dv,rank", [(3, 128, 128, 64), (2, 64, 64, 64), (2, 128, 128, 32), (5, 64, 64, 32)])
@pytest.mark.parametrize("spoiled", [False, True])
def test_gated_delta_norm_forms_its_gates(lens, H, D, Dv, rank, spoiled, monkeypatch):
    """the gate formed behind the norm against the gate as a step of its own: the same three-part product in another order, the same fp32
    norm - one bf16 ulp where a rounding falls the other way; an infinite or undefined projection spoils its own token and head only"""
    from scratchpad_amd import _native
    announce("gated delta lowrank norm", lens, H, D, Dv, rank, spoiled)
    monkeypatch.setattr(_native, "delta_chunks_pay", lambda *a: True)
    g = torch.Generator(device=DEV).manual_seed(21)
    T, slots = sum(lens), slots_of(lens)
    q, k, v, bp, p = torch.randn(T, 2 * H * D + H * Dv + 8 * H + rank, generator=g, device=DEV).bfloat16().split([H * D, H * D, H * Dv, 8 * H, rank], 1)
    bp, p = bp[:, :H], p.clone()
    w2t = torch.randn(rank, H * Dv, generator=g, device=DEV) * rank ** -0.5 * 2
    if spoiled:
        p[3, 1], p[7, 0] = float("inf"), float("nan")
        w2t[2, 5] = float("inf")
    decay, nw = torch.rand(T, H * D, generator=g, device=DEV), torch.rand(Dv, generator=g, device=DEV) + 0.5
    outs = []
    for gate in ((p, w2t), _native.lowrank_gate(p, w2t, None, "sigmoid")):
        S = torch.zeros(2 * len(lens) + 1, H, D, Dv, device=DEV)
        outs.append(_native.gated_delta_scan(q, k, v, bp, decay, gate, nw, S, seq_extend(lens, [0] * len(lens), slots), H, H, D, Dv, 1e-5).float())
    got, want = outs
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isfinite(want).any()
    ok = torch.isfinite(want)
    assert ((got - want).abs()[ok] <= 2.0 ** -7 * want.abs()[ok] + 1e-6).all() and (got != want)[ok].float().mean() < 0.01


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_steps_without_requests(dtype):
    """every recurrence takes a multi-token step of no request: no rows, no state moved"""
    from scratchpad_amd import _native as nat
    H, D = 2, 64
    n = H * D
    ints = lambda dt: torch.zeros(0, dtype=dt, device=DEV)  # noqa: E731
    seq = nat.SeqParams(ints(torch.int64), ints(torch.int64), ints(torch.int32), ints(torch.int32), ints(torch.int32),
                        torch.zeros(0, dtype=torch.int32, device=DEV))
    x = lambda w=n, dt=dtype: torch.zeros(0, w, dtype=dt, device=DEV)  # noqa: E731
    f32 = lambda *s: torch.ones(*s, device=DEV)  # noqa: E731
    S, m = f32(1, H, D, D), f32(1, H)
    outs = [nat.mamba2_scan(x(3 * n), x(H, torch.float32), f32(H), f32(H), f32(H), S, seq, H, H, D, D),
            nat.mlstm_scan(x(), x(), x(), x(), x(H, torch.float32), x(H, torch.float32), f32(n), S, f32(1, H, D), m, seq, H, D, D, 15.0, 1e-5),
            nat.delta_recurrence(x(), x(), x(), x(), x(n, torch.float32), x(n, torch.float32), f32(n), S, seq, H, D, 1e-5),
            nat.hgrn2_scan(x(), x(), x(), f32(n), f32(n), f32(D), S, seq, H, D, D, 1e-5),
            nat.gated_delta_scan(x(), x(), x(), x(H), x(n, torch.float32), (x(32), f32(32, n)), f32(D), S, seq, H, H, D, D, 1e-5),
            nat.gated_delta_scan(x(), x(), x(), x(H), x(n, torch.float32), x(n, torch.float32), f32(D), S, seq, H, H, D, D, 1e-5)]
    torch.cuda.synchronize()
    assert all(o.shape == (0, n) for o in outs) and bool((S == 1).all()) and bool((m == 1).all())
