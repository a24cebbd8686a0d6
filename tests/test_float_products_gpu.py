"""Products of 32-bit operands on the matrix cores against double precision, at the edges of the kernels'
tiles, and beside the kernel on the vector ALU."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(a, w, epi, c0):
    y = a.double() @ w.double().T
    if epi == 1:
        return c0.double() + y
    if epi == 2:
        g, u = y[:, 0::2], y[:, 1::2]
        return g / (1 + torch.exp(-g)) * u
    return y


def operands(M, N, K, epi, seed=0):
    gen = torch.Generator(device=DEV).manual_seed(seed + M * 7 + N)
    a = torch.randn(M, K, generator=gen, device=DEV)
    w = torch.randn(N, K, generator=gen, device=DEV) / K ** 0.5
    c = torch.randn(M, N // 2 if epi == 2 else N, generator=gen, device=DEV)
    return a, w, c


# up to 16 rows the staged kernel (16, 24, 32 and 48 weight rows a workgroup), then tiles of 32, 64 and
# 128 rows, whole and cut along K; one row more and less than each; widths that end inside a tile
@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 130, 257])
@pytest.mark.parametrize("N,K", [(6, 32), (130, 96), (2048, 2048), (6144, 256), (12282, 64), (16384, 96), (1000, 8192)])
def test_float_product(M, N, K):
    from picolm_amd import kernels
    for epi in (0, 1, 2):
        a, w, c = operands(M, N, K, epi)
        ref = reference(a, w, epi, c)
        kernels.gemm(a, w, c, epi)
        # sums of K products of unit variance in all: rounding errors of 2^-24 a step add in quadrature
        # (and worst cases of M N of them lie five standard deviations out); silu multiplies by up to |u|
        bound = 6.0 * 2 ** -24 * K ** 0.5 * max(1.0, float(ref.abs().max())) + 4e-7 * float(ref.abs().max())
        assert float((c - ref).abs().max()) <= bound, (M, N, K, epi, float((c - ref).abs().max()), bound)


@pytest.mark.parametrize("M,N,K", [(4, 2048, 8192), (24, 3072, 2048), (60, 2048, 8192), (460, 2048, 8192), (460, 16384, 2048)])
def test_float_product_is_no_less_precise_than_the_vector_alu(M, N, K):
    from picolm_amd import kernels
    a, w, c = operands(M, N, K, 0)
    ref, there = reference(a, w, 0, c), torch.empty_like(c)
    kernels.gemm(a, w, c, 0)
    kernels.gemm_generic(a, w, there, 0)
    error = lambda x: float((x - ref).norm() / ref.norm())
    print(f"{M} x {N} x {K}: {error(c):.3e} beside {error(there):.3e}")
    assert error(c) <= 1.05 * error(there)


def test_float_product_other_operands_keep_the_vector_alu():
    """K no multiple of 32, rows that do not start at 16 bytes, a bfloat16 operand."""
    from picolm_amd import kernels
    for M, N, K in ((5, 70, 45), (70, 40, 40)):
        a, w, c = operands(M, N, K, 0)
        ref = reference(a, w, 0, c)
        kernels.gemm(a, w, c, 0)
        assert float((c - ref).abs().max()) <= 1e-5
    a, w, c = operands(9, 64, 64, 0)
    shifted = torch.empty(9 * 64 + 1, device=DEV)[1:].view(9, 64).copy_(a)
    kernels.gemm(shifted, w, c, 0)
    assert float((c - reference(a, w, 0, c)).abs().max()) <= 1e-5
    kernels.gemm(a, w.bfloat16(), c, 0)
    assert float((c - reference(a, w.bfloat16(), 0, c)).abs().max()) <= 1e-5


def test_float_product_of_a_row_does_not_depend_on_the_other_rows():
    """The staged kernel, every tile height, and products cut into their shares sum in one order."""
    from picolm_amd import kernels
    for N, K in ((2048, 2048), (300, 8192), (4100, 96), (16384, 320)):
        for epi in (0, 1, 2):
            a, w, c = operands(700, N, K, epi)
            want = c.clone()
            kernels.gemm(a, w, want, epi)
            for M in (1, 5, 16, 20, 33, 64, 100, 200, 460):
                got = c[:M].clone()
                kernels.gemm(a[:M].contiguous(), w, got, epi)
                assert torch.equal(got, want[:M]), (M, N, K, epi)


def test_float_products_on_two_streams():
    """Products that are cut into shares at the same time on two streams: each has partial sums of its own."""
    from picolm_amd import kernels
    streams, work = [torch.cuda.Stream() for _ in range(2)], []
    for i in range(2):
        a, w, c = operands(40, 2048, 8192, 0, seed=i)
        want = torch.empty_like(c)
        kernels.gemm(a, w, want, 0)
        work.append((a, w, want, [torch.empty_like(c) for _ in range(20)]))
    torch.cuda.synchronize()
    for k in range(20):
        for s, (a, w, want, outs) in zip(streams, work):
            with torch.cuda.stream(s):
                kernels.gemm(a, w, outs[k], 0)
    torch.cuda.synchronize()
    for a, w, want, outs in work:
        assert all(torch.equal(o, want) for o in outs)
