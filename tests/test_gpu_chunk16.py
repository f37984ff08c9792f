"""The recurrences that run 16 tokens at a time with their operands formed beforehand: requests whose lengths lie around the chunk's and the
segment's edges, from an empty and from a held state, against the token-by-token recurrence in 64 bits.  Everything is fp32 in both: the
states differ by accumulated fp32 roundings - the sums over 16 tokens and D channels and a product of decays per chunk - 2e-5 of the largest
value being ten times that; outputs by a few roundings of the terms they are summed from (the head's norm amplifies them where a row nearly
cancels) and one rounding of their type."""
import pytest
import torch

from tests.test_gpu_toredra_kernels import DEV, announce, seq_extend

pytestmark = pytest.mark.gpu
LENS = [[1], [15, 16, 17], [48, 1, 33, 2], [16, 200, 3], [40] + [2] * 66 + [20]]
HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}


def near(got, want, bar=2e-5):
    assert torch.isfinite(got).all()
    err = (got.double() - want).abs().max() / want.abs().max()
    assert err <= bar, f"{err:.2e} > {bar:.0e}"


def near_rows(got, want, size, dtype, bar=3e-6):
    """one rounding of the type, and a share of the absolute terms of a read-out's sum: the largest seen over these cases is 7e-7 (fp32)"""
    assert torch.isfinite(got.float()).all()
    rounding = (HALF[dtype] * want.abs()).clamp_min(2.0 ** -25 if dtype == torch.float16 else 0.0)      # (halves below 2^-14 are equally far apart)
    over = ((got.double() - want).abs() - rounding) / size.clamp_min(1e-30)
    assert float(over.max()) <= bar, f"{float(over.max()):.2e} > {bar:.0e}"


def rms(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def hgrn2_reference(q, f, v, fb, lower, S, H):
    """(normed read-outs, the same of the sums' absolute terms, state)"""
    T, D, Dv = q.shape[0], q.shape[1] // H, v.shape[1] // H
    q, f, v, lo = q.double(), f.double(), v.double().view(T, H, Dv), lower.double()
    q, w = (q * torch.sigmoid(q)).view(T, H, D), (lo + (1 - lo) * torch.sigmoid(f + fb.double())).view(T, H, D)
    o, size = (torch.empty(T, H, Dv, dtype=torch.float64, device=DEV) for _ in range(2))
    for t in range(T):
        S = w[t][:, :, None] * S + (1 - w[t])[:, :, None] * v[t][:, None]
        o[t], size[t] = (S * q[t][:, :, None]).sum(1), (S * q[t][:, :, None]).abs().sum(1)
    return rms(o), size / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5), S


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("segment", [0, 16, 64])
@pytest.mark.parametrize("lens", LENS, ids=lambda l: "-".join(map(str, l[:5])))
@pytest.mark.parametrize("H,D,Dv", [(2, 128, 128), (3, 64, 64), (1, 128, 64), (2, 64, 128)])
def test_hgrn2_chunks(lens, H, D, Dv, segment, dtype, monkeypatch):
    from scratchpad_amd import _native
    announce("hgrn2 chunks", dtype, lens, H, D, Dv, segment)
    monkeypatch.setattr(_native, "SCAN_SEGMENT", segment)
    monkeypatch.setattr(_native, "HGRN2_CHUNKS", True)
    g = torch.Generator(device=DEV).manual_seed(7)
    T, slots = sum(lens), [2 * i + 1 for i in range(len(lens))]
    S = torch.full((2 * len(lens) + 1, H, D, Dv), float("nan"), device=DEV)
    fb, lower, nw = torch.randn(H * D, generator=g, device=DEV), torch.rand(H * D, generator=g, device=DEV) * 0.5, torch.rand(Dv, generator=g, device=DEV) + 0.5
    ref = [torch.zeros(H, D, Dv, dtype=torch.float64, device=DEV) for _ in lens]
    for prefixes in ([0] * len(lens), lens):                     # the second launch goes on from what the first one left
        a = (torch.randn(T, 2 * H * D + H * Dv, generator=g, device=DEV) * 2).to(dtype)
        q, f, v = a.split([H * D, H * D, H * Dv], 1)
        out = _native.hgrn2_scan(q, f, v, fb, lower, nw, S, seq_extend(lens, prefixes, slots), H, D, Dv, 1e-5).view(T, H, Dv)
        at = 0
        for i, n in enumerate(lens):
            want, size, ref[i] = hgrn2_reference(q[at:at + n], f[at:at + n], v[at:at + n], fb, lower, ref[i], H)
            near(S[slots[i]], ref[i])
            near_rows(out[at:at + n], want * nw.double(), size * nw.double(), dtype)
            at += n
    assert torch.isnan(S[::2]).all()                             # no other slot was touched


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["query", "forget", "value"])
@pytest.mark.parametrize("at", [0, 5, 15, 16, 50])
def test_hgrn2_numbers_that_are_not_finite_reach_no_earlier_token(at, where, bad, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "SCAN_SEGMENT", 32)
    monkeypatch.setattr(_native, "HGRN2_CHUNKS", True)
    H, D, T = 2, 64, 70
    g = torch.Generator(device=DEV).manual_seed(8)
    a = torch.randn(T, 3 * H * D, generator=g, device=DEV).bfloat16()
    zero, one = torch.zeros(H * D, device=DEV), torch.ones(D, device=DEV)

    def run(a):
        S = torch.zeros(2, H, D, D, device=DEV)
        out = _native.hgrn2_scan(*a.split(H * D, 1), zero, zero, one, S, seq_extend([T], [0], [1]), H, D, D, 1e-5)
        return out.view(T, H, D), S[1]
    clean = run(a)
    b = a.clone()
    b[at, {"query": 0, "forget": H * D, "value": 2 * H * D}[where] + 3] = bad
    out, S = run(b)
    assert torch.equal(out[:at], clean[0][:at]) and torch.equal(out[:, 1], clean[0][:, 1]) and torch.equal(S[1], clean[1][1])
    # what is finite is what the recurrence token by token leaves finite (an infinite pre-activation of the gate: all)
    monkeypatch.setattr(_native, "HGRN2_CHUNKS", False)
    ref, ref_S = run(b)
    assert torch.equal(out.isfinite(), ref.isfinite()) and torch.equal(S.isfinite(), ref_S.isfinite())
    ok = ref.isfinite()
    assert ((out - ref).float().abs()[ok] <= 2.0 ** -7 * ref.float().abs()[ok] + 1e-5).all()
    assert ok.all() == (where == "forget" and bad == float("inf")) and ok[at + 1:].all() == (where == "query" or bool(ok.all()))


def delta_reference(r, k, v, g, w, a, S, H):
    """as hgrn2_reference, gated"""
    T, D = r.shape[0], r.shape[1] // H
    r, k, v, g, w, a = (x.double().view(T, H, D) for x in (r, k, v, g, w, a))
    o, size = (torch.empty(T, H, D, dtype=torch.float64, device=DEV) for _ in range(2))
    for t in range(T):
        u = k[t] / torch.sqrt((k[t] * k[t]).sum(-1, keepdim=True) + 1e-6)
        y = (S * u[:, :, None]).sum(1)
        S = w[t][:, :, None] * S - (a[t] * u)[:, :, None] * y[:, None] + k[t][:, :, None] * v[t][:, None]
        o[t], size[t] = (S * r[t][:, :, None]).sum(1), (S * r[t][:, :, None]).abs().sum(1)
    gate = torch.sigmoid(g)
    return rms(o) * gate, size / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * gate, S


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lens", LENS, ids=lambda l: "-".join(map(str, l[:5])))
@pytest.mark.parametrize("H,D", [(3, 64), (1, 64)])
def test_delta_recurrence_chunks(lens, H, D, dtype, monkeypatch):
    from scratchpad_amd import _native
    announce("delta recurrence chunks", dtype, lens, H, D)
    monkeypatch.setattr(_native, "DELTA_RECURRENCE_CHUNKS", True)
    gen = torch.Generator(device=DEV).manual_seed(9)
    T, slots = sum(lens), [2 * i + 1 for i in range(len(lens))]
    S = torch.full((2 * len(lens) + 1, H, D, D), float("nan"), device=DEV)
    nw = torch.rand(H * D, generator=gen, device=DEV) + 0.5
    ref = [torch.zeros(H, D, D, dtype=torch.float64, device=DEV) for _ in lens]
    for prefixes in ([0] * len(lens), lens):
        r, k, v, g = torch.randn(T, 4 * H * D, generator=gen, device=DEV).to(dtype).split(H * D, 1)
        w = torch.exp(-0.6 * torch.rand(T, H * D, generator=gen, device=DEV))
        a = torch.rand(T, H * D, generator=gen, device=DEV)
        out = _native.delta_recurrence(r, k, v, g, w, a, nw, S, seq_extend(lens, prefixes, slots), H, D, 1e-5).view(T, H, D)
        at = 0
        for i, n in enumerate(lens):
            rows = slice(at, at + n)
            want, size, ref[i] = delta_reference(r[rows], k[rows], v[rows], g[rows], w[rows], a[rows], ref[i], H)
            near(S[slots[i]], ref[i])
            near_rows(out[rows], want * nw.double().view(H, D), size * nw.double().view(H, D), dtype)
            at += n
    assert torch.isnan(S[::2]).all()


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["read", "key", "value", "decay", "remove"])
@pytest.mark.parametrize("at", [0, 5, 15, 16, 50])
def test_delta_numbers_that_are_not_finite_reach_no_earlier_token(at, where, bad, monkeypatch):
    from scratchpad_amd import _native
    monkeypatch.setattr(_native, "DELTA_RECURRENCE_CHUNKS", True)
    H, D, T = 2, 64, 70
    gen = torch.Generator(device=DEV).manual_seed(10)
    x = [torch.randn(T, H * D, generator=gen, device=DEV).bfloat16() for _ in range(4)]
    x += [torch.exp(-0.6 * torch.rand(T, H * D, generator=gen, device=DEV)), torch.rand(T, H * D, generator=gen, device=DEV)]

    def run(x):
        S = torch.zeros(2, H, D, D, device=DEV)
        out = _native.delta_recurrence(*x, torch.ones(H * D, device=DEV), S, seq_extend([T], [0], [1]), H, D, 1e-5)
        return out.view(T, H, D), S[1]
    clean = run(x)
    y = [t.clone() for t in x]
    y[{"read": 0, "key": 1, "value": 2, "decay": 4, "remove": 5}[where]][at, 3] = bad
    out, S = run(y)
    assert torch.equal(out[:at], clean[0][:at]) and torch.equal(out[:, 1], clean[0][:, 1]) and torch.equal(S[1], clean[1][1])
    monkeypatch.setattr(_native, "DELTA_RECURRENCE_CHUNKS", False)
    ref, ref_S = run(y)
    assert torch.equal(out.isfinite(), ref.isfinite()) and torch.equal(S.isfinite(), ref_S.isfinite())
    ok = ref.isfinite()
    assert ((out - ref).float().abs()[ok] <= 2.0 ** -7 * ref.float().abs()[ok] + 1e-5).all()
    assert not ok.all() and ok[at + 1:].all() == (where == "read")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens", [[70], [5, 33, 200]], ids=lambda l: "-".join(map(str, l)))
@pytest.mark.parametrize("rule", ["hgrn2", "delta"])
def test_decays_of_zero_one_and_next_to_nothing(rule, lens, dtype, monkeypatch):
    """products of decays that vanish or underflow, which quotients of them would not survive: HGRN2's gates closed and open to the last
    bit, the delta rule's decays 0, 1e-30, 1e-38 (two of them: none in fp32) and 1"""
    from scratchpad_amd import _native
    announce("extreme decays", rule, lens, dtype)
    monkeypatch.setattr(_native, "HGRN2_CHUNKS", True)
    monkeypatch.setattr(_native, "DELTA_RECURRENCE_CHUNKS", True)
    monkeypatch.setattr(_native, "SCAN_SEGMENT", 64)
    gen = torch.Generator(device=DEV).manual_seed(14)
    H, D, T, n = 2, 64, sum(lens), 2 * 64
    slots = list(range(1, len(lens) + 1))
    S = torch.randn(len(lens) + 1, H, D, D, generator=gen, device=DEV)
    start, seq = S.double(), seq_extend(lens, [3] * len(lens), slots)
    x = torch.randn(T, 4 * n, generator=gen, device=DEV).to(dtype)
    pick = torch.randint(0, 4, (T, n), generator=gen, device=DEV)
    if rule == "hgrn2":
        f = torch.tensor([-200.0, 200.0, -60.0, 0.5], device=DEV)[pick].to(dtype)
        q, v, zero = x[:, :n], x[:, n:2 * n], torch.zeros(n, device=DEV)
        out = _native.hgrn2_scan(q, f, v, zero, zero, torch.ones(D, device=DEV), S, seq, H, D, D, 1e-5).view(T, H, D)
    else:
        w = torch.tensor([0.0, 1e-30, 1e-38, 1.0], device=DEV)[pick]
        w[:, ::3] = 1.0
        a = torch.rand(T, n, generator=gen, device=DEV)
        out = _native.delta_recurrence(*x.split(n, 1), w, a, torch.ones(n, device=DEV), S, seq, H, D, 1e-5).view(T, H, D)
    at = 0
    for i, m in enumerate(lens):
        rows = slice(at, at + m)
        if rule == "hgrn2":
            want, size, end = hgrn2_reference(q[rows], f[rows], v[rows], zero, zero, start[i + 1], H)
        else:
            want, size, end = delta_reference(*(t[rows] for t in x.split(n, 1)), w[rows], a[rows], start[i + 1], H)
        near(S[i + 1], end)
        near_rows(out[rows], want, size, dtype, 1e-5)
        at += m


WINDOW_LENS = [[400], [130, 0, 16, 1, 250], [5] * 40 + [200, 33], [17] * 300]


def window_problem(H, cols, lens, seed):
    """heads so many that a step of these lengths takes several passes over the workspace; half of the requests hold a state"""
    from scratchpad_amd import _native
    g = torch.Generator(device=DEV).manual_seed(seed)
    T, prefixes, slots = sum(lens), [(3 * i) % 2 * 7 for i in range(len(lens))], list(range(1, len(lens) + 1))
    return g, T, seq_extend(lens, prefixes, slots), len(lens) + 1, _native


@pytest.mark.parametrize("lens", WINDOW_LENS, ids=lambda l: "-".join(map(str, l[:5])))
def test_delta_recurrence_in_passes_over_a_bounded_workspace(lens, monkeypatch):
    """1024 heads: 9 chunks a pass; the heads' bits are those of the same heads in a step of one pass"""
    H, D, sub = (128 if len(lens) > 100 else 1024), 64, 2
    g, T, seq, slots, nat = window_problem(H, D, lens, 31)
    announce("delta recurrence in passes", lens[:5], H)
    monkeypatch.setattr(nat, "DELTA_RECURRENCE_CHUNKS", True)
    floats = nat.load().sp_delta_recurrence_chunk_floats
    assert 4 * floats(T, len(lens), H, D) <= (192 << 20) + 12 * len(lens) * 200 < 4 * 5376 * H * (T // 16 + len(lens))
    rows = torch.randn(T, 4 * H * D, generator=g, device=DEV).bfloat16()
    w = torch.exp(-0.6 * torch.rand(T, H * D, generator=g, device=DEV))
    a, nw = torch.rand(T, H * D, generator=g, device=DEV), torch.rand(H * D, generator=g, device=DEV) + 0.5
    S = torch.randn(slots, H, D, D, generator=g, device=DEV)
    start = S.clone()
    out = nat.delta_recurrence(*rows.split(H * D, 1), w, a, nw, S, seq, H, D, 1e-5)
    assert torch.equal(S[0], start[0])
    for h in (0, H // 2 - 1, H - sub):
        cut = slice(h * D, (h + sub) * D)
        part = start[:, h:h + sub].contiguous()
        few = nat.delta_recurrence(*(x[:, cut] for x in rows.split(H * D, 1)), w[:, cut].contiguous(), a[:, cut].contiguous(), nw[cut].contiguous(),
                                   part, seq, sub, D, 1e-5)
        assert torch.isfinite(few.float()).all() and torch.equal(out[:, cut], few) and torch.equal(S[:, h:h + sub], part)


@pytest.mark.parametrize("lens", WINDOW_LENS, ids=lambda l: "-".join(map(str, l[:5])))
@pytest.mark.parametrize("segment", [0, 64])
def test_hgrn2_in_passes_over_a_bounded_workspace(lens, segment, monkeypatch):
    """512 heads of 128: 21 chunks a pass; bit for bit without segments, with them within their own roundings"""
    H, D, sub = (64 if len(lens) > 100 else 512), 128, 2
    g, T, seq, slots, nat = window_problem(H, D, lens, 32)
    announce("hgrn2 in passes", lens[:5], H, segment)
    monkeypatch.setattr(nat, "HGRN2_CHUNKS", True)
    assert 4 * nat.load().sp_hgrn2_chunk_floats(T, len(lens), H, D) <= (192 << 20) + 12 * len(lens) * 200 < 4 * 4608 * H * (T // 16 + len(lens))
    rows = torch.randn(T, 3 * H * D, generator=g, device=DEV).bfloat16()
    fb, lower = torch.randn(H * D, generator=g, device=DEV), torch.rand(H * D, generator=g, device=DEV) * 0.5
    nw, S = torch.rand(D, generator=g, device=DEV) + 0.5, torch.randn(slots, H, D, D, generator=g, device=DEV)
    start = S.clone()
    monkeypatch.setattr(nat, "SCAN_SEGMENT", segment)
    out = nat.hgrn2_scan(*rows.split(H * D, 1), fb, lower, nw, S, seq, H, D, D, 1e-5)
    assert torch.equal(S[0], start[0])
    monkeypatch.setattr(nat, "SCAN_SEGMENT", 0)
    for h in (0, H // 2 - 1, H - sub):
        cut = slice(h * D, (h + sub) * D)
        part = start[:, h:h + sub].contiguous()
        few = nat.hgrn2_scan(*(x[:, cut] for x in rows.split(H * D, 1)), fb[cut].contiguous(), lower[cut].contiguous(), nw, part, seq, sub, D, D, 1e-5)
        if segment == 0:
            assert torch.isfinite(few.float()).all() and torch.equal(out[:, cut], few) and torch.equal(S[:, h:h + sub], part)
        else:
            near(S[:, h:h + sub], part.double())
            assert ((out[:, cut].double() - few.double()).abs() <= 2 * HALF[torch.bfloat16] * few.double().abs() + 1e-3).all()
