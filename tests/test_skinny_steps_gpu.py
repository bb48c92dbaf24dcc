"""The weight-streaming product's steps of K, waves a workgroup and activation
(csrc/skinny_gemm.hip) against 64 bits, and what lies beside its operands."""
import pytest
import torch

import kubeai_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operands(M, N, K, seed):
    torch.manual_seed(seed)
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    return x, torch.randn(N, K, device=DEV, dtype=torch.bfloat16)


def _near_gated(y, x, w, gelu):
    """2^-8 of the result for its rounding; the products' fp32 sums within 2^-13 of
    their magnitudes, times the other factor (an activation's slope is under 1.2)."""
    (g, u), (e, f) = (x.double() @ w.double().T).chunk(2, -1), (
        2.0 ** -13 * (x.double().abs() @ w.double().abs().T)).chunk(2, -1)
    fn = torch.nn.functional
    right = (fn.gelu(g, approximate="tanh") if gelu else fn.silu(g)) * u
    tol = 2.0 ** -8 * right.abs() + 1.2 * e * u.abs() + f * (g.abs() + 1.2 * e) + 1e-5
    assert ((y.double() - right).abs() <= tol).all()


# K: 1 to 7 steps of 128 values, whole and not; N: 8, 4 and 2 waves, ends in a wave
@pytest.mark.parametrize("K", [32, 128, 160, 256, 384, 416, 544, 896])
@pytest.mark.parametrize("N", [8, 24, 200, 18432, 16384, 28680])
def test_gated(N, K):
    for M in (1, 7, 16):
        x, w = _operands(M, N, K, M + N + K)
        y = torch.full((M, N // 2), 7.0, device=DEV, dtype=torch.bfloat16)
        for act in (1, 2):
            ops._C.skinny_gated(y, x, w, act)
            _near_gated(y, x, w, act == 2)


@pytest.mark.parametrize("M,N,K", [(3, 16384, 160), (16, 28672, 288), (9, 18448, 96),
                                   (5, 384, 1312), (40, 384, 1312)])
def test_neighbours_stay_out(M, N, K):
    """Bytes past the operands' ends, and rows of no finite values beside a row of
    finite ones, do not reach its results."""
    x, w = _operands(M, N, K, 1)
    want = (x.double() @ w.double().T).float()
    bad_x, bad_w = x.clone(), w.clone()
    bad_x[1], bad_w[N // 2] = float("inf"), float("nan")
    # the operands in front of what must not be read
    bad_x, bad_w = (torch.cat([t, torch.full_like(t[:32], float("nan"))])[: t.shape[0]]
                    for t in (bad_x, bad_w))
    y = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    ops._C.skinny_linear(y, bad_x, bad_w, None, None, None)
    rows, cols = torch.arange(M) != 1, torch.arange(N) != N // 2
    got, want = y[rows][:, cols].float(), want[rows][:, cols]
    # fp32 sums and one rounding
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -13 * (x.abs().double() @ w.abs().double().T)[rows][:, cols]
    assert ((got - want).abs() <= tol).all()
    assert not y[1].isfinite().any() and y[:, N // 2].isnan().all()


@pytest.mark.parametrize("M", [17, 40, 64, 96])
@pytest.mark.parametrize("fp8", [False, True])
def test_few_rows_of_the_tiled_product(M, fp8):
    """Workgroups that begin at columns of K apart."""
    N, K = 24576, 4096 if fp8 else 2048
    assert ops._tiled_better(M, N, K, fp8)
    x, w = _operands(M, N, K, M)
    if fp8:
        (x, sx), (w, sw) = ops.quant_fp8(x), ops.quant_fp8(w)
        y = ops.linear_fp8(x, sx, w, sw.view(1, -1))
        x, w = x.double() * sx[:, None].double(), w.double() * sw[:, None].double()
    else:
        y = ops.linear(x, w)
    want = x.double() @ w.double().T
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -13 * (x.double().abs() @ w.double().abs().T)
    assert ((y.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("N,K,fp8", [(18432, 128, True), (18448, 256, True), (24592, 384, True),
                                     (32752, 1408, True), (65536, 64, False),
                                     (65552, 192, False), (65536, 2112, False)])
@pytest.mark.parametrize("M", [17, 96])
def test_few_rows_of_few_steps(M, N, K, fp8):
    """The tiled product of fewer steps of K than its first columns are apart, through
    the calls that choose it."""
    assert ops._tiled_better(M, N, K, fp8)
    x, w = _operands(M, N, K, M)
    if fp8:
        (x, sx), (w, sw) = ops.quant_fp8(x), ops.quant_fp8(w)
        y = ops.linear_fp8(x, sx, w, sw.view(1, -1))
        x, w = x.double() * sx[:, None].double(), w.double() * sw[:, None].double()
    else:
        y = ops.linear(x, w)
    want = x.double() @ w.double().T
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -13 * (x.double().abs() @ w.double().abs().T)
    assert ((y.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("T", [1, 16, 17, 40, 96])
@pytest.mark.parametrize("gelu", [False, True])
def test_activation_goes_with_few_rows(T, gelu):
    x, w = _operands(T, 28672, 2048, T)
    y = ops.gated(x, w, gelu)
    assert y is not None
    _near_gated(y, x, w, gelu)
    with torch.enable_grad():
        assert ops.gated(x.requires_grad_(), w, gelu) is None


def test_activation_goes_where_linear_streams():
    for N, K, here in ((49152, 1280, True), (16384, 8192, True), (16384 - 16, 2048, False)):
        assert ops._streams_better(8, N, K, fp8=False) is here
        x, w = _operands(8, N, K, N)
        y = ops.gated(x, w)
        assert (y is not None) is here
        if here:
            _near_gated(y, x, w, False)


@pytest.mark.parametrize("M,N,K,fp8,better", [
    # us, library / streaming
    (8, 16384, 4096, False, True),     # 32.1 / 23.7
    (1, 128256, 4096, False, True),    # 185 / 168
    (16, 28672, 4096, True, True),     # 32.0 / 23.9
    (8, 9216, 6656, True, True),       # 37.6 / 18.9
    (16, 8192, 8192, True, False),     # 16.4 / 21.3
    (8, 14848, 7680, False, False),    # 45 / 52
    (8, 256000, 2304, False, False),   # 207 / 218
    (11, 59648, 9472, True, False),    # 102 / 112
    (8, 65536, 128, True, False),      # 5.6 / 6.7
    (17, 28672, 4096, True, False),    # (the tiled product's)
])
def test_rule(M, N, K, fp8, better):
    assert ops._streams_better(M, N, K, fp8) is better
