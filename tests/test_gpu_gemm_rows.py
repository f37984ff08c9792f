"""The three forms of sp_gemm_skinny (1 row, 2-4 rows, 5-16 rows) at the edges of their tiles: columns that leave a remainder in a
workgroup, rows of K that end inside a wave's loads, the rows where one form takes over from the next, views with strides, an
unguarded tail behind the output, and subnormal operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def run(x, w, N, epilogue, out):
    from scratchpad_amd import _native
    _native._check(_native.load().sp_gemm_skinny(out.data_ptr(), x.data_ptr(), w.data_ptr(), x.shape[0], N, x.shape[1], x.stride(0),
                                                 w.stride(0), out.stride(0), epilogue, _native._dt(x), _native._stream()), "sp_gemm_skinny")


def bound(ref, x, w, eps):
    # one rounding of the result, and fp32 sums of K products in any order: K * 2^-24 of the sum of their magnitudes
    return eps * ref.abs() + x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-45


@pytest.mark.parametrize("dtype,eps", [(torch.bfloat16, 2.0 ** -8), (torch.float16, 2.0 ** -11)])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("N,K", [(1, 32), (7, 96), (9, 480), (24, 2080), (37, 8224), (2, 4128), (2048, 544), (2049, 1056), (2051, 2080), (4099, 2048)])
def test_rows_columns_and_lengths(dtype, eps, M, N, K):
    g = torch.Generator().manual_seed(M * 31 + N * 7 + K)
    big = torch.randn(M, K + 64, generator=g).to(dtype).cuda()
    x = big[:, 32:32 + K]                                             # rows with a stride, 16-byte aligned
    wide = (torch.randn(N, K + 8, generator=g) * 0.05).to(dtype).cuda()
    w = wide[:, :K]
    out = torch.full((M + 1, N + 3), 7.0, dtype=dtype, device="cuda")
    run(x, w, N, 0, out)
    xc, wc = x.cpu(), w.cpu()
    ref = xc.double() @ wc.double().T
    assert bool(((out[:M, :N].cpu().double() - ref).abs() <= bound(ref, xc, wc, eps)).all())
    assert bool((out[M:] == 7.0).all()) and bool((out[:, N:] == 7.0).all())          # nothing written past the result
    run(x, w, N, 2, out)                                              # max(., 0)^2 of the fp32 sum
    err = (out[:M, :N].cpu().double() - ref.clamp(min=0).square()).abs()
    slack = K * 2.0 ** -24 * (xc.double().abs() @ wc.double().abs().T)
    # subnormal halves keep 2^-25 of absolute precision
    assert bool((err <= eps * (ref.clamp(min=0) + slack).square() + 2 * (ref.abs() + slack) * slack + 2.0 ** -25).all())


@pytest.mark.parametrize("M", [2, 3, 6])
@pytest.mark.parametrize("N,K", [(130, 512), (130, 544), (2304, 1536), (2304, 4064), (2304, 4096), (2304, 4128), (4104, 1536), (4104, 1568)])
def test_both_sides_of_the_lines_between_the_forms(M, N, K):
    test_rows_columns_and_lengths(torch.bfloat16, 2.0 ** -8, M, N, K)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("I,K", [(1, 32), (6, 96), (13, 2080), (1024, 544), (1030, 1024), (2049, 2048)])
@pytest.mark.parametrize("epilogue", [1, 3])
def test_gate_times_up_has_the_bits_of_its_two_steps(dtype, M, I, K, epilogue):
    from scratchpad_amd import _native
    g = torch.Generator().manual_seed(M + I + K)
    x = torch.randn(M, K, generator=g).to(dtype).cuda()
    w = (torch.randn(2 * I, K, generator=g) * 0.2).to(dtype).cuda()
    both = torch.empty(M, 2 * I, dtype=dtype, device="cuda")
    run(x, w, 2 * I, 0, both)
    got = torch.empty(M, I, dtype=dtype, device="cuda")
    run(x, w, I, epilogue, got)
    assert torch.equal(got, (_native.silu_and_mul if epilogue == 1 else _native.gelu_tanh_and_mul)(both))


@pytest.mark.parametrize("dtype,tiny,eps", [(torch.bfloat16, 2.0 ** -130, 2.0 ** -8), (torch.float16, 2.0 ** -20, 2.0 ** -11)])
@pytest.mark.parametrize("M", [1, 3, 9])
def test_subnormal_operands_count(dtype, tiny, eps, M):
    g = torch.Generator().manual_seed(M)
    x = (torch.randint(-8, 9, (M, 256), generator=g).double() * tiny).to(dtype)
    w = (torch.randint(-8, 9, (16, 256), generator=g).double() * 16).to(dtype)
    out = torch.empty(M, 16, dtype=dtype, device="cuda")
    run(x.cuda(), w.cuda(), 16, 0, out)
    ref = x.double() @ w.double().T                                   # whole multiples of tiny: the sums are exact in fp32
    floor = 2.0 ** -134 if dtype == torch.bfloat16 else 2.0 ** -25    # half of the smallest step of the result's type
    assert bool(((out.cpu().double() - ref).abs() <= eps * ref.abs() + floor).all())
