"""Pairs ordered by expert, and the choice of experts, at the edges of their kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def nat():
    from scratchpad_amd import _native
    return _native


@pytest.mark.parametrize("pairs", [1, 63, 1025, 16384, 16385, 40000])
@pytest.mark.parametrize("experts", [1, 32, 64, 65, 1000, 4096])
def test_pairs_are_ordered_by_expert(nat, pairs, experts):
    """registers up to 16384 pairs, `place` above; sums over experts in runs of 64"""
    g = torch.Generator().manual_seed(pairs + experts)
    ids = torch.randint(0, experts, (pairs,), generator=g, dtype=torch.int32)
    if pairs == 1025:
        ids[:] = experts - 1                                            # all in one
    offsets, order, place = (t.cpu().long() for t in nat.moe_align(ids.to(DEV).view(-1, 1), experts))
    count = torch.bincount(ids.long(), minlength=experts)
    assert torch.equal(offsets, torch.cat([torch.zeros(1, dtype=torch.long), count.cumsum(0)]))
    assert torch.equal(order.sort().values, torch.arange(pairs)) and torch.equal(order[place], torch.arange(pairs))
    assert torch.equal(ids.long()[order], torch.repeat_interleave(torch.arange(experts), count))


@pytest.mark.parametrize("experts", [5, 32, 64, 65, 200])
@pytest.mark.parametrize("ties", [False, True])
def test_largest_choices_win_and_the_lower_index_among_equal_ones(nat, experts, ties):
    """scores to a few roundings of 64 bits (one exponential and one sum of at most 200 terms); which experts exactly"""
    g = torch.Generator().manual_seed(experts)
    z = torch.randint(-2, 3, (70, experts), generator=g).float() if ties else torch.randn(70, experts, generator=g)
    z[1] = -3.0                                                         # all equal
    z[2, : experts - 4] = float("-inf")                                 # as many as are wanted
    top = 4
    logits, ids = z.to(DEV), torch.empty(70, top, dtype=torch.int32, device=DEV)
    weights = torch.empty(70, top, dtype=torch.float32, device=DEV)
    assert nat.load().sp_moe_softmax_topk(ids.data_ptr(), weights.data_ptr(), None, logits.data_ptr(), experts, None, 70, experts, top, 1, 1,
                                          1.0, 0, torch.cuda.current_stream().cuda_stream) == 0
    score = z.double().softmax(-1)
    # choices are compared in 32 bits: equal logits have equal scores there, and random ones lie further apart than their rounding
    want = torch.sort(z, dim=-1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), want)
    assert torch.allclose(weights.cpu().double(), score.gather(1, want), rtol=300 * 2.0 ** -24, atol=0)
