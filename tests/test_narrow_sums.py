"""Sums of up to 64 rows in tiles of 64 columns, and where they are taken."""
import pytest
import torch

from kubeai_amd import ops


@pytest.mark.parametrize("M,N,K,fp8,better", [
    (40, 4096, 4096, True, True), (40, 4096, 14336, True, True),
    (1, 4096, 4096, False, True), (64, 2304, 9216, False, True),
    (65, 4096, 4096, True, False), (0, 4096, 4096, True, False),
    (40, 6144, 4096, True, True), (40, 6144, 4096, False, False),  # 192 workgroups
    (8, 2048, 2048, True, False),                                 # two steps each
    (16, 4096, 2560, True, False), (17, 4096, 2560, True, True),  # five
    (8, 8256, 8192, False, False), (8, 16384, 4224, True, True), (8, 16448, 4096, True, False),
    # eight parts
    (32, 2048, 8192, True, False), (33, 2048, 8192, True, True), (1, 2048, 4096, False, False),
    (33, 2048, 4096, False, True), (1, 2112, 4608, False, True),
    # one part
    (8, 16384, 4096, True, False), (40, 16384, 4096, True, False), (1, 14336, 8192, False, False),
    (16, 14336, 9088, False, True), (17, 14336, 9088, False, False), (17, 14336, 8064, True, True),
    (17, 14336, 8320, True, False), (16, 14336, 8320, True, True), (1, 8192, 4224, False, True),
    # two to seven
    (16, 8192, 4096, False, False), (17, 8192, 4096, False, True), (1, 4096, 4096, False, True),
    (16, 4096, 16384, True, False), (17, 4096, 16384, True, True), (49, 7168, 14976, True, True),
    (49, 7168, 15104, True, False), (48, 7168, 15104, True, True),
])
def test_where_they_are_taken(M, N, K, fp8, better):
    assert ops.narrow_better(M, N, K, fp8) is better


def _operands(M, N, K, fp8, seed):
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(M, K, generator=g).bfloat16(), torch.randn(N, K, generator=g).bfloat16()
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    return x.cuda(), w.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 63, 64])
@pytest.mark.parametrize("N,K", [(16, 128), (64, 256), (80, 2176), (4080, 1152), (2304, 2048),
                                 (4096, 1280), (16384, 256), (16400, 128)])
@pytest.mark.parametrize("fp8", [False, True])
def test_sums(M, N, K, fp8):
    """Last tiles of few columns, parts of unlike lengths, fewer steps than parts and
    than places in LDS, one part."""
    x, w = _operands(M, N, K, fp8, M + N)
    part = ops._C.narrow_sums(x, w)
    assert part.shape[1:] == (M, N) and 1 <= part.shape[0] <= 8
    want = x.double() @ w.double().t()
    # what the matrix instructions keep of the terms they add (test_tiled_linear_gpu.py)
    size = x.double().abs() @ w.double().abs().t()
    assert ((part.double().sum(0) - want).abs() <= 2.0 ** -13 * size).all()
    assert torch.equal(part, ops._C.narrow_sums(x, w))  # the same bits each time


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
def test_rows_that_are_no_numbers_stay_apart(fp8):
    x, w = _operands(40, 4096, 2048, fp8, 5)
    x = x.clone()
    x[7, 100] = float("nan")
    got = ops._C.narrow_sums(x, w).sum(0)
    bad = got.isnan().any(1)
    assert bad[7] and bad.sum() == 1


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 40, 64])
@pytest.mark.parametrize("fp8", [False, True])
def test_readers(M, fp8):
    """The norm of the product that sums_for_reader gives, and the routes not taken."""
    N, K = 4096, 4096
    x, w = _operands(M, N, K, fp8, 9)
    sx = torch.rand(M, device="cuda") / K ** 0.5 + 0.01 if fp8 else None
    sw = torch.rand(1, N, device="cuda") + 0.5 if fp8 else None
    sums = ops.sums_for_reader(x, w, sx, sw.view(-1) if fp8 else None)
    assert torch.equal(sums.part, ops._C.narrow_sums(x, w))
    norm = torch.rand(N, device="cuda").bfloat16()
    got = ops.rmsnorm(sums, norm, 1e-5).double()
    y = x.double() @ w.double().t()
    if fp8:
        y = y * sx.double()[:, None] * sw.double()
    want = y * torch.rsqrt(y.square().mean(1, keepdim=True) + 1e-5) * norm.double()
    # the product's and the result's roundings to bf16
    assert (got - want).norm() < 4e-3 * want.norm()
    assert ops.tiled_sums(x, w[:, : K - 64]) is None
    with pytest.raises(RuntimeError):
        ops._C.narrow_sums(x[:1].expand(65, -1).contiguous(), w)
