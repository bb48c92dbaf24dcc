"""Tiled products of many rows (csrc/tiled_gemm.h) with every tile shape, one to
five steps of K (the places in LDS are two to four), whole and in parts, rows
and columns one off a tile, and which operands go to the library.

Against the product in 64 bits: rounding to the 8 significant bits of bf16
moves a result by at most 2^-8 of itself, fp32 sums of K <= 2048 terms by at
most 2^-13 of the sum of the terms' sizes; two scales are two more fp32 products."""
import pytest
import torch

import kubeai_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# rows, columns, steps of K
SIZES = [(1, 16, 1), (63, 272, 2), (65, 528, 3), (129, 144, 4), (100, 400, 5), (1, 16, 16),
         (193, 8208, 1), (385, 8208, 2), (385, 12304, 3), (900, 12304, 2), (900, 8208, 4), (1025, 8208, 3),
         (1025, 8208, 5), (1500, 8208, 5), (2049, 6160, 2), (2048, 6144, 3), (700, 16, 16)]


def _operands(M, N, steps, fp8):
    torch.manual_seed(M + N + steps)
    K = steps * (128 if fp8 else 64)
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(N, K, device=DEV, dtype=torch.bfloat16)
    if not fp8:
        return x, w, None, None
    return (x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn),
            torch.rand(M, device=DEV) + 0.1, torch.rand(N, device=DEV) + 0.1)


def _reference(x, w, sx, sw):
    a, b = x.double(), w.double()
    y, size = a @ b.T, a.abs() @ b.abs().T
    if sx is not None:
        s = sx[:, None].double() * sw.double()
        y, size = y * s, size * s
    return y, size


@pytest.mark.parametrize("M,N,steps", SIZES)
@pytest.mark.parametrize("fp8", [False, True])
def test_tiled_products(M, N, steps, fp8):
    from kubeai_amd import _C

    x, w, sx, sw = _operands(M, N, steps, fp8)
    want, size = _reference(x, w, sx, sw)
    y = torch.full((M + 1, N), 7.0, device=DEV, dtype=torch.bfloat16)
    _C.tiled_linear(y[:M], x, w, sx, sw, 0)
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -13 * size
    assert ((y[:M].double() - want).abs() <= tol + 1e-30).all()
    assert (y[M] == 7).all()
    part = _C.tiled_sums(x, w)
    assert part.shape[1:] == (M, N) and part.dtype == torch.float32
    got = part.double().sum(0)
    if fp8:
        got = got * sx[:, None].double() * sw.double()
    assert ((got - want).abs() <= 2.0 ** -13 * size + 1e-30).all()


@pytest.mark.parametrize("M,N,steps", [(1, 16, 1), (63, 144, 2), (129, 400, 5), (385, 8208, 3),
                                       (1500, 8208, 2), (2049, 6160, 3)])
@pytest.mark.parametrize("fp8,act", [(False, 1), (True, 1), (False, 2)])
def test_activations_of_gate_and_up(M, N, steps, fp8, act):
    """silu' and gelu' are within [-0.2, 1.2] and |silu(g)|, |gelu(g)| <= |g|: an
    error of e in gate and f in up moves the result by at most 1.2 e |u| + f |g| and
    their product; the exponential and the division are right to a few units of
    2^-22 (times the exponent, |y| < 30 here, where the result counts)."""
    from kubeai_amd import _C

    x, w, sx, sw = _operands(M, N, steps, fp8)
    if fp8:
        sw *= w.shape[1] ** -0.5
    else:
        w *= w.shape[1] ** -0.5
    want, size = _reference(x, w, sx, sw)
    (g, u), (e, f) = want.chunk(2, -1), (2.0 ** -13 * size).chunk(2, -1)
    y = torch.empty(M, N // 2, device=DEV, dtype=torch.bfloat16)
    _C.tiled_linear(y, x, w, sx, sw, act)
    fn = torch.nn.functional
    right = (fn.silu(g) if act == 1 else fn.gelu(g, approximate="tanh")) * u
    tol = 2.0 ** -8 * right.abs() + 1.2 * e * u.abs() + f * (g.abs() + 1.2 * e) + 1e-5
    assert ((y.double() - right).abs() <= tol).all()
    # the same among experts
    c = torch.tensor([M // 3, 0, M - M // 3], device=DEV, dtype=torch.int32)
    stack = w.view(torch.uint8).expand(3, N, -1).contiguous().view(w.dtype)
    got = ops.grouped_linear(x, stack, c, act=act,
                             scales=(sx, sw.expand(3, N).contiguous()) if fp8 else None)
    assert ((got.double() - right).abs() <= tol).all()


def test_sizes_reach_every_shape():
    from kubeai_amd import _C

    for sums in (False, True):
        plans = [_C.tiled_plan(M, N, steps * 128, fp8, sums)
                 for M, N, steps in SIZES for fp8 in (False, True)]
        assert {p[0] for p in plans} == set(range(8))
        assert any(p[1] > 1 for p in plans) == sums


@pytest.mark.parametrize("N", [4, 20, 1028])
def test_columns_that_are_no_units_of_eight(N):
    from kubeai_amd import _C

    x, w, _, _ = _operands(130, N, 3, False)
    want, size = _reference(x, w, None, None)
    y = torch.empty(130, N, device=DEV, dtype=torch.bfloat16)
    _C.tiled_linear(y, x, w, None, None, 0)
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * size).all()
    got = _C.tiled_sums(x, w).double().sum(0)
    assert ((got - want).abs() <= 2.0 ** -13 * size).all()


def test_infinities_and_nan_stay_in_their_rows_and_columns():
    from kubeai_amd import _C

    x, w, _, _ = _operands(300, 272, 3, False)
    x[7, 5], w[19, 5], x[280, 100] = float("inf"), 1.0, float("nan")
    y = torch.empty(300, 272, device=DEV, dtype=torch.bfloat16)
    _C.tiled_linear(y, x, w, None, None, 0)
    assert y[280].isnan().all() and not y[7].isfinite().any() and y[7, 19] == float("inf")
    rest = torch.ones(300, dtype=torch.bool)
    rest[[7, 280]] = False
    assert y[rest.to(DEV)].isfinite().all()


def test_routes_of_fp8_products():
    """Forms that the tiled product does not take give the library's result:
    strided rows, a bias, a result that is a slice, too few columns of K."""
    x, w, sx, sw = _operands(700, 2048, 16, True)
    want, _ = _reference(x, w, sx, sw)

    def near(y, add=0.0):
        torch.testing.assert_close(y.double(), want + add, atol=2e-2, rtol=2.0 ** -7)

    assert ops._tiled_operands(x, w)
    near(ops.linear_fp8(x, sx, w, sw.view(1, -1)))
    out = torch.empty(700, 2048, device=DEV, dtype=torch.bfloat16)
    assert ops.linear_fp8(x, sx, w, sw.view(1, -1), out=out) is out
    near(out)
    b = torch.randn(2048, device=DEV, dtype=torch.bfloat16)
    near(ops.linear_fp8(x, sx, w, sw.view(1, -1), b), b.double())
    wide = torch.zeros(700, 2048 + 128, device=DEV, dtype=torch.uint8).view(x.dtype)
    wide[:, :2048] = x
    assert not ops._tiled_operands(wide[:, :2048], w)
    near(ops.linear_fp8(wide[:, :2048], sx, w, sw.view(1, -1)))
    odd = torch.zeros(2048 * 2048 + 1, device=DEV, dtype=torch.uint8)[1:].view(2048, 2048)
    odd = odd.view(w.dtype).copy_(w)
    assert not ops._tiled_operands(x, odd)
    assert not ops._tiled_operands(x[:, :64].contiguous(), w[:, :64].contiguous())
    assert not ops._tiled_operands(x, w[:2040])  # (the library refuses these columns)
