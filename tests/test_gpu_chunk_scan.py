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
