"""Extend launches with few row blocks: half blocks and keys shared over workgroups against the oracle and the general form."""
import pytest
import torch

from oracle import ops
from tests.helpers import DTYPES, assert_attn_close, cpu
from tests.test_gpu_attention import extend_problem

pytestmark = pytest.mark.gpu
DEV = "cuda"
# (prefix, new) per request: one tile and a key more, a single token, a request without new tokens, more shares than tiles, odd row blocks
PRE, EXT = [1000, 0, 64, 700, 5], [65, 1, 0, 130, 300]


@pytest.fixture(scope="module")
def nat():
    from scratchpad_amd import _native
    return _native


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 64), (6, 3, 64), (3, 3, 64), (16, 2, 128), (5, 5, 128), (12, 2, 128)])
def test_forms_of_small_extend_launches(nat, dt, kv8, causal, Hq, Hkv, D):
    """Half blocks (heads of 64) and shares are held to one unit of the error model that every attention kernel is held to (their sums are
    the same 32-bit sums in another order); the plan, or its absence, changes no bit; too small a workspace gives the form that needs none."""
    dtype = DTYPES[dt]
    p, q, ext, start = extend_problem(91, Hq, Hkv, D, PRE, EXT, dtype)
    if kv8:
        for name in ("k_buffer", "v_buffer"):
            p[name] = p[name].float().to(torch.float8_e5m2).view(torch.uint8)
    if not causal:
        p["seq_lens"][1] = 0                                       # no key at all: zeros
    plan = nat.extend_plan(ext, p["seq_lens"], sum(EXT), Hq, Hkv, causal)
    full = nat.extend_workspace_bytes(sum(EXT), len(EXT), Hq, D, dtype)

    def run(form, planned, nbytes=full):
        ws, o = torch.full((nbytes + 4096,), 0xff, dtype=torch.uint8, device=DEV), torch.full_like(q, float("nan"))
        try:
            nat.debug_set("extend_small", form)
            nat.extend_attention(o, q, p["k_buffer"], p["v_buffer"], p["req_to_token"], p["req_pool_indices"], p["seq_lens"], ext, start,
                                 D ** -0.5, 0.0, causal, max(EXT), int(p["seq_lens"].max()), ws[:nbytes], plan=plan if planned else None)
            torch.cuda.synchronize()
        finally:
            nat.debug_set("extend_small", 0)
        assert bool((ws[nbytes:] == 0xff).all()), "nothing written past the workspace"
        return o

    c = cpu(p)
    pools = [c[n].view(torch.float8_e5m2).float() if kv8 else c[n].float() for n in ("k_buffer", "v_buffer")]
    oracle = lambda v: ops.extend_attention(q.cpu().float(), pools[0], v, c["req_to_token"], c["req_pool_indices"], c["seq_lens"], ext.cpu(),
                                            start.cpu(), D ** -0.5, causal=causal)
    ref, aref = oracle(pools[1]), oracle(pools[1].abs())
    general, half = run(1, True), run(2, True)
    assert torch.equal(general, half) == (D != 64), "form 2: half blocks, which add in another order, where they exist"
    for form in (0, 1, 2, 3, 6, 17):
        o = run(form, True)
        assert torch.equal(o, run(form, False)), f"form {form}: the plan decides the order only"
        assert_attn_close(o, ref, aref, dtype, what=f"extend form {form}")
        assert form != 1 or torch.equal(o, general)
        assert torch.equal(run(form, True, 12 * sum(EXT) + 64), general if form == 1 else half), f"form {form} without room for shares"


def test_values_that_are_not_finite_reach_the_rows_that_see_them(nat):
    """an infinite and a missing value in one share: rows that see the key carry them on, the others don't"""
    pre, ext_l = [900], [40]
    p, q, ext, start = extend_problem(92, 4, 1, 64, pre, ext_l, torch.bfloat16)
    slot = p["req_to_token"][int(p["req_pool_indices"][0])]
    p["v_buffer"][int(slot[100]), 0, 3] = float("inf")
    p["v_buffer"][int(slot[900 + 20]), 0, 5] = float("nan")
    ws = torch.empty(nat.extend_workspace_bytes(40, 1, 4, 64, torch.bfloat16), dtype=torch.uint8, device=DEV)
    outs = []
    for form in (1, 5):
        o = torch.zeros_like(q)
        try:
            nat.debug_set("extend_small", form)
            nat.extend_attention(o, q, p["k_buffer"], p["v_buffer"], p["req_to_token"], p["req_pool_indices"], p["seq_lens"], ext, start, 0.125,
                                 0.0, True, 40, 940, ws)
        finally:
            nat.debug_set("extend_small", 0)
        outs.append(o)
    assert bool((outs[0][:, :, 3] == float("inf")).all())
    assert torch.equal(outs[0].isfinite(), outs[1].isfinite()) and torch.equal(outs[0].isnan(), outs[1].isnan())


def test_shares_replay_in_a_graph(nat):
    """the plan, the lengths and the workspace are read at replay: eager results after each replay, with other work between"""
    pre, ext_l = [1500, 300], [50, 30]
    p, q, ext, start = extend_problem(93, 32, 8, 64, pre, ext_l, torch.bfloat16)
    ws = torch.empty(nat.extend_workspace_bytes(80, 2, 32, 64, torch.bfloat16), dtype=torch.uint8, device=DEV)
    args = (q, p["k_buffer"], p["v_buffer"], p["req_to_token"], p["req_pool_indices"], p["seq_lens"], ext, start, 0.125, 0.0, True, 50, 1550, ws)
    ref, out = torch.zeros_like(q), torch.zeros_like(q)
    nat.extend_attention(ref, *args)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        nat.extend_attention(out, *args)
    for _ in range(3):
        out.fill_(float("nan"))
        ws.fill_(0xff)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("Hq,Hkv", [(8, 2), (6, 3), (3, 3)])
@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("pre,new", [([1000, 0, 64, 700, 5], [65, 1, 0, 130, 300]), ([0, 63, 64], [64, 1, 65]), ([511, 448], [1, 64])])
def test_tiles_shared_by_the_halves_of_a_workgroup(nat, dt, causal, Hq, Hkv, kv8, pre, new):
    """heads of 64: even and odd tiles by four waves each - one tile, odd counts, a half without a visible tile, no key at all"""
    dtype, D = DTYPES[dt], 64
    p, q, ext, start = extend_problem(17, Hq, Hkv, D, pre, new, dtype)
    if kv8:
        for name in ("k_buffer", "v_buffer"):
            p[name] = p[name].float().to(torch.float8_e5m2).view(torch.uint8)
    if not causal:
        p["seq_lens"][0] = 0
    ws = torch.empty(nat.extend_workspace_bytes(sum(new), len(new), Hq, D, dtype), dtype=torch.uint8, device=DEV)
    plan = nat.extend_plan(ext, p["seq_lens"], sum(new), Hq, Hkv, causal)
    outs = []
    try:
        nat.debug_set("extend_small", 2)
        for pl in (plan, None):
            o = torch.full_like(q, float("nan"))
            nat.extend_attention(o, q, p["k_buffer"], p["v_buffer"], p["req_to_token"], p["req_pool_indices"], p["seq_lens"], ext, start, D ** -0.5,
                                 0.0, causal, max(new), int(p["seq_lens"].max()), ws, plan=pl)
            outs.append(o)
    finally:
        nat.debug_set("extend_small", 0)
    c = cpu(p)
    keys, values = (c[n].view(torch.float8_e5m2).float() if kv8 else c[n].float() for n in ("k_buffer", "v_buffer"))
    oracle = lambda v: ops.extend_attention(q.cpu().float(), keys, v, c["req_to_token"], c["req_pool_indices"],  # noqa: E731
                                            c["seq_lens"], ext.cpu(), start.cpu(), D ** -0.5, causal=causal)
    assert torch.equal(outs[0], outs[1])
    assert_attn_close(outs[0], oracle(values), oracle(values.abs()), dtype, what=f"half blocks {pre} {new}")
