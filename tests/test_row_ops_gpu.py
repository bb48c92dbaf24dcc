"""Row kernels at the edges of their splits (256, 512 and up to 1024 threads
a row, 1 to 8 units of 8 values a thread, rows below and above 1024) and the
fused rotation and cache write against the two-kernel route.

Bounds: bf16 outputs are rounded once (2^-9 of themselves; the norm's fp32
sum adds below 1e-5). fp8 outputs: a value may land on the neighbouring
eight-bit number where the fp32 quotient differs in its last bits, 2^-3 of
itself, in less than one value in 500; the scale is fp32."""
import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.engine.quant import Fp8Linear
from kubeai_amd.ops import ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
WIDTHS = [8, 504, 512, 2048, 4096, 4104, 8192, 16384]


def _x(T, H):
    torch.manual_seed(T * 7 + H)
    return torch.randn(T, H, device=DEV, dtype=torch.bfloat16)


def _close_fp8(q, s, want):
    """q * s against want [T, H] fp32."""
    amax = want.abs().amax(-1).clamp_min(1e-6)
    torch.testing.assert_close(s, amax / 448.0, atol=0, rtol=1e-5)
    exact = (want / (amax / 448.0)[:, None]).to(torch.float8_e4m3fn).float()
    off = q.float() != exact
    assert off.float().mean().item() < 2e-3
    torch.testing.assert_close(q.float(), exact, atol=2.0 ** -9, rtol=2.0 ** -3 + 1e-6)


@pytest.mark.parametrize("H", WIDTHS)
@pytest.mark.parametrize("T", [1, 3, 1023, 1024])
def test_norms(T, H):
    x, r = _x(T, H), _x(T + 1, H)[1:].contiguous()
    w = torch.randn(H, device=DEV, dtype=torch.bfloat16)
    want = ref.rmsnorm(x.float(), w.float(), 1e-5)
    torch.testing.assert_close(ops.rmsnorm(x, w, 1e-5).float(), want, atol=1e-5, rtol=2.0 ** -8)
    _close_fp8(*ops.rmsnorm_fp8(x, w, 1e-5), want)
    want, total = ref.fused_add_rmsnorm(x.float(), r.float(), w.float(), 1e-5)
    r2 = r.clone()
    _close_fp8(*ops.fused_add_rmsnorm_fp8(x, r2, w, 1e-5), want)
    assert torch.equal(r2, total.bfloat16())
    got, r3 = ops.fused_add_rmsnorm(x.clone(), r.clone(), w, 1e-5)
    torch.testing.assert_close(got.float(), want, atol=1e-5, rtol=2.0 ** -8)
    assert torch.equal(r3, r2)


@pytest.mark.parametrize("H", WIDTHS + [14336, 28672, 32768])
@pytest.mark.parametrize("T", [1, 1024])
def test_to_fp8(T, H):
    x = _x(T, H)
    _close_fp8(*ops.quant_fp8(x), x.float())
    gu = _x(T, 2 * H)
    g, u = gu.float().chunk(2, -1)
    q, s = ops.silu_and_mul_fp8(gu)
    # __expf: 2 ulp around 1 + e^-g
    _close_fp8(q, s, torch.nn.functional.silu(g) * u)


def test_zero_and_huge_rows():
    x = torch.zeros(4, 512, device=DEV, dtype=torch.bfloat16)
    x[1] = 3e38
    x[2, 5] = 1e-30
    q, s = ops.quant_fp8(x)
    assert (q[0].float() == 0).all() and (q[1].float() == 448).all()
    torch.testing.assert_close(s[:1], torch.full((1,), 1e-6 / 448, device=DEV))


@pytest.mark.parametrize("nq,nkv,hd", [(32, 8, 128), (3, 1, 16), (8, 4, 256), (5, 5, 80)])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e5m2])
@pytest.mark.parametrize("pad", [0, 8])
def test_rope_and_cache_equals_two_kernels(nq, nkv, hd, cache, pad):
    T, width = 21, (nq + 2 * nkv) * hd
    qkv = _x(T, width + pad)[:, :width]
    pos = torch.randint(0, 900, (T,), device=DEV, dtype=torch.int32)
    slots = torch.randperm(5 * 16, device=DEV)[:T]
    slots[3] = -1
    cs = ref.make_cos_sin_cache(hd, 1000).to(DEV)
    one = [torch.zeros(5, nkv, 16, hd, device=DEV).to(cache) for _ in range(2)]
    two = [c.clone() for c in one]
    other = qkv.clone()
    q = ops.rope_and_cache(qkv, nq, pos, cs, *one, slots)
    q2, k2, v2 = other.split([nq * hd, nkv * hd, nkv * hd], -1)
    q2, k2 = ops.rope(q2.unflatten(-1, (nq, hd)), k2.unflatten(-1, (nkv, hd)), pos, cs)
    ops.reshape_and_cache(k2, v2.unflatten(-1, (nkv, hd)), *two, slots)
    # the compiler may contract x1 c - x2 s either way: the fp32 values differ in
    # their last bit and fall to different sides of a rounding tie about once in
    # 2^15 values (bf16); then by one step of the result's type
    step = 2.0 ** -7 if cache == torch.bfloat16 else 2.0 ** -2
    for a, b, rtol in [(q, q2, 2.0 ** -7)] + [(a, b, step) for a, b in zip(one, two)]:
        a, b = a.float(), b.float()
        assert (a != b).sum().item() <= 2 + a.numel() // 1000
        torch.testing.assert_close(a, b, atol=1e-6, rtol=rtol)
    assert torch.equal(one[1].view(torch.uint8), two[1].view(torch.uint8))


@pytest.mark.parametrize("M", [1, 17, 96])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("N,K", [(512, 1024), (4112, 512), (1008, 9216)])
def test_norms_of_product_sums(M, fp8, N, K):
    """Added on the way in, the parts give the same bf16 row as added first; the
    norms of the two may contract their fp32 products either way, which moves
    one output in some hundreds by one step of its type."""
    from kubeai_amd import _C

    def near(a, b, step):
        a, b = a.float(), b.float()
        assert (a != b).sum().item() <= 2 + a.numel() // 100
        torch.testing.assert_close(a, b, atol=1e-6, rtol=step)

    x, w = _x(M, K), _x(N, K) * 0.05
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(M, device=DEV) + 0.5, torch.rand(N, device=DEV) + 0.5
    y = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    _C.skinny_linear(y, x, w, sx, sw, None)
    weight = torch.randn(N, device=DEV, dtype=torch.bfloat16)
    r = _x(M, N)

    def sums():
        p = ops.product_sums(x, w, sx, sw)
        assert isinstance(p, ops.ProductSums)
        return p

    near(ops.rmsnorm(sums(), weight, 1e-5), ops.rmsnorm(y, weight, 1e-5), 2.0 ** -7)
    (a, sa), (b, sb) = ops.rmsnorm_fp8(sums(), weight, 1e-5), ops.rmsnorm_fp8(y, weight, 1e-5)
    near(a, b, 2.0 ** -3)
    torch.testing.assert_close(sa, sb, atol=0, rtol=1e-6)
    r1, r2 = r.clone(), r.clone()
    got, res = ops.fused_add_rmsnorm(sums(), r1, weight, 1e-5)
    want, _ = ops.fused_add_rmsnorm(y.clone(), r2, weight, 1e-5)
    assert res is r1 and torch.equal(r1, r2)
    near(got, want, 2.0 ** -7)
    r1, r2 = r.clone(), r.clone()
    (a, sa), (b, sb) = (ops.fused_add_rmsnorm_fp8(sums(), r1, weight, 1e-5),
                        ops.fused_add_rmsnorm_fp8(y, r2, weight, 1e-5))
    near(a, b, 2.0 ** -3)
    torch.testing.assert_close(sa, sb, atol=0, rtol=1e-6)
    assert torch.equal(r1, r2)


@pytest.mark.parametrize("T", [256, 257, 1023, 1024])
@pytest.mark.parametrize("H", [4096, 4104, 8192, 16384])
@pytest.mark.parametrize("fp8", [False, True])
def test_norms_of_sums_of_many_rows(T, H, fp8):
    """On both sides of 256 and 1024 rows, where the threads of a row change: the row is
    the parts' sum in bf16, whatever they are."""
    torch.manual_seed(T + H)
    part = torch.randn(3, T, H, device=DEV)
    sx, sw = torch.rand(T, device=DEV) + 0.5, torch.rand(H, device=DEV) + 0.5
    weight = torch.randn(H, device=DEV, dtype=torch.bfloat16)
    r = _x(T, H)
    h = part[0] + part[1] + part[2]
    if fp8:
        h = h * sx[:, None] * sw
    want, total = ref.fused_add_rmsnorm(h.bfloat16().float(), r.float(), weight.float(), 1e-5)
    sums = ops.ProductSums(part, *((sx, sw) if fp8 else (None, None)))
    if fp8:
        (q, s), res = ops.fused_add_rmsnorm_fp8(sums, r, weight, 1e-5), r
        _close_fp8(q, s, want)
    else:
        out, res = ops.fused_add_rmsnorm(sums, r, weight, 1e-5)
        torch.testing.assert_close(out.float(), want, atol=1e-6, rtol=2.0 ** -8)
    assert torch.equal(res, total.bfloat16())


@pytest.mark.parametrize("M", [1, 40, 1030])
@pytest.mark.parametrize("N", [8, 520, 2304, 16384])
def test_branch_norm_add_and_norm(M, N):
    """One launch has the bits of the three that it replaces."""
    x, r = _x(M, N), _x(M, N)
    w1, w2 = (torch.randn(N, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    kept = r.clone()

    out, hidden = ops.add_and_norm(x, r, w2, 1e-5)
    assert torch.equal(hidden, x + r) and torch.equal(r, kept)
    assert torch.equal(out, ops.rmsnorm(x + r, w2, 1e-5))
    out, hidden = ops.add_and_norm(ops.BranchNorm(x, w1, 1e-5), r, w2, 1e-5)
    assert torch.equal(hidden, r + ops.rmsnorm(x, w1, 1e-5))
    assert torch.equal(out, ops.rmsnorm(hidden, w2, 1e-5))
    # forms that the launch does not take go one by one
    wide = torch.cat([r, r], 1)[:, :N]
    out2, hidden2 = ops.add_and_norm(x, wide, w2, 1e-5) if N == 8 else (out, hidden)
    if N == 8:
        assert torch.equal(hidden2, x + r)
        assert torch.equal(out2, ops.rmsnorm(hidden2, w2, 1e-5))
    if M <= 96 and 512 <= N <= 4096 and N % 16 == 0:
        a, w = _x(M, 1024), _x(N, 1024) * 0.05
        y = ops.rmsnorm(ops.product_sums(a, w), w1, 1e-5)
        out, hidden = ops.add_and_norm(
            ops.BranchNorm(ops.product_sums(a, w), w1, 1e-5), r, w2, 1e-5)
        assert torch.equal(hidden, r + y)
        assert torch.equal(out, ops.rmsnorm(hidden, w2, 1e-5))


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("cache", [torch.bfloat16, torch.float8_e5m2])
def test_rope_of_product_sums(fp8, cache):
    from kubeai_amd import _C

    T, nq, nkv, hd, K = 21, 6, 2, 64, 1024
    width = (nq + 2 * nkv) * hd
    x, w = _x(T, K), _x(width, K) * 0.05
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(T, device=DEV) + 0.5, torch.rand(width, device=DEV) + 0.5
    y = torch.empty(T, width, device=DEV, dtype=torch.bfloat16)
    _C.skinny_linear(y, x, w, sx, sw, None)
    pos = torch.randint(0, 900, (T,), device=DEV, dtype=torch.int32)
    slots = torch.randperm(32, device=DEV)[:T]
    slots[2] = -1
    cs = ref.make_cos_sin_cache(hd, 1000).to(DEV)
    one = [torch.zeros(2, nkv, 16, hd, device=DEV).to(cache) for _ in range(2)]
    two = [c.clone() for c in one]
    q = ops.rope_and_cache(ops.product_sums(x, w, sx, sw), nq, pos, cs, *one, slots)
    q2 = ops.rope_and_cache(y, nq, pos, cs, *two, slots)
    assert q.is_contiguous()
    step = 2.0 ** -7 if cache == torch.bfloat16 else 2.0 ** -2  # see above
    for a, b, rtol in [(q, q2, 2.0 ** -7)] + [(a, b, step) for a, b in zip(one, two)]:
        a, b = a.float(), b.float()
        assert (a != b).sum().item() <= 2 + a.numel() // 1000
        torch.testing.assert_close(a, b, atol=1e-6, rtol=rtol)


def test_linear_routes_agree():
    """Shapes on both sides of every rule, against the library's product."""
    for M, N, K in [(1, 16384, 64), (16, 16384, 64), (17, 16384, 64), (3, 16368, 64),
                    (96, 1024, 16384), (97, 1024, 16384), (5, 2048, 16384), (8, 65552, 64)]:
        x, w = _x(M, K), _x(N, K) * K ** -0.5
        want = torch.nn.functional.linear(x.float(), w.float())
        torch.testing.assert_close(ops.linear(x, w).float(), want, atol=2e-3, rtol=2.0 ** -7)
        x8, w8 = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(M, device=DEV) + 0.5, torch.rand(1, N, device=DEV) + 0.5
        b = torch.randn(N, device=DEV, dtype=torch.bfloat16)
        want = torch.nn.functional.linear(x8.float(), w8.float()) * sx[:, None] * sw + b.float()
        got = ops.linear_fp8(x8, sx, w8, sw, b)
        # the library adds the bias in fp32 or after rounding, as it likes
        torch.testing.assert_close(got.float(), want, atol=2e-2, rtol=2.0 ** -7)


def test_products_of_operands_that_begin_anywhere():
    """A slice of one row counts as contiguous whatever its address and stride;
    the kernels that read 16 bytes at a time leave it to the library."""
    torch.manual_seed(3)
    N, K = 512, 17408
    w = torch.randn(N, K, device=DEV, dtype=torch.bfloat16) * K ** -0.5
    odd = torch.empty(N * K + 1, device=DEV, dtype=torch.bfloat16)[1:].view(N, K).copy_(w)
    wide = torch.randn(3, K + 9, device=DEV, dtype=torch.bfloat16)
    for x, m in ((wide[:1, 1 : K + 1], w), (wide[:1, :K], w), (wide[:, :K].contiguous(), odd)):
        want = torch.nn.functional.linear(x.float(), m.float())
        torch.testing.assert_close(ops.linear(x, m).float(), want, atol=2e-3, rtol=2.0 ** -7)
        assert ops.product_sums(x, m) is None
    x = wide[:1, 1 : K + 1]
    lin = Fp8Linear(w)
    torch.testing.assert_close(lin(x).float(), lin(x.clone()).float(), atol=2e-2, rtol=2.0 ** -6)


def test_products_under_transforms():
    """What follows operations sees the product: forward mode, vmap, a trace,
    autocast, a dispatch mode, and gradients of the input."""
    import torch.autograd.forward_ad as fwd
    from torch.utils.flop_counter import FlopCounterMode

    torch.manual_seed(4)
    N, K = 20480, 256  # a width that few rows go through the streaming kernel at
    w = torch.randn(N, K, device=DEV, dtype=torch.bfloat16) * K ** -0.5
    x, t = _x(4, K), _x(4, K) * 0.5
    want, slope = torch.nn.functional.linear(x, w), torch.nn.functional.linear(t, w)

    def near(a, b):
        torch.testing.assert_close(a.float(), b.float(), atol=2e-3, rtol=2.0 ** -6)

    with fwd.dual_level():
        y = fwd.unpack_dual(ops.linear(fwd.make_dual(x, t), w))
        near(y.primal, want)
        assert y.tangent is not None
        near(y.tangent, slope)
    near(torch.func.jvp(lambda v: ops.linear(v, w), (x,), (t,))[1], slope)
    near(torch.func.vmap(lambda v: ops.linear(v, w))(torch.stack([x, t]))[1], slope)
    traced = torch.jit.trace(lambda v: ops.linear(v, w), (x,))
    near(traced(t), slope)
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w).dtype == torch.float16
    with FlopCounterMode(display=False) as flops:
        ops.linear(x, w)
    assert flops.get_total_flops() == 2 * 4 * N * K
    v = x.clone().requires_grad_()
    ops.linear(v, w).float().sum().backward()
    near(v.grad, w.float().sum(0).expand(4, K))
    lin = Fp8Linear(w)
    assert lin(v).requires_grad and not lin(x).requires_grad


@pytest.mark.parametrize("parts", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 15, 17])
@pytest.mark.parametrize("N,scaled", [(520, True), (4096, False), (8200, True)])
def test_any_number_of_parts(parts, N, scaled):
    """Whatever is left of the eights that are added at once, and with scales or none:
    the bits of the parts added in order in fp32, scaled by row and column, rounded."""
    T, hd = 19, 8
    torch.manual_seed(parts)
    part = torch.randn(parts, T, N, device=DEV)
    sx = torch.rand(T, device=DEV) + 0.5 if scaled else None
    sw = (torch.rand(N + 1, device=DEV) + 0.5)[1:] if scaled else None  # 4 bytes off
    y = torch.zeros(T, N, device=DEV)
    for p in part:
        y = y + p
    y = (y * sx[:, None] * sw if scaled else y).to(torch.bfloat16)
    w, r = torch.randn(N, device=DEV, dtype=torch.bfloat16), _x(T, N)
    got, res = ops.fused_add_rmsnorm(ops.ProductSums(part, sx, sw), r.clone(), w, 1e-5)
    want, kept = ops.fused_add_rmsnorm(y.clone(), r.clone(), w, 1e-5)
    assert torch.equal(res, kept) and torch.equal(res, y + r)
    torch.testing.assert_close(got, want, atol=0, rtol=2.0 ** -7)  # a step: contractions
    _, hidden = ops.add_and_norm(
        ops.BranchNorm(ops.ProductSums(part, sx, sw), w, 1e-5), r, w, 1e-5)
    torch.testing.assert_close(hidden, r + ops.rmsnorm(y, w, 1e-5), atol=2.0 ** -7, rtol=2.0 ** -7)
    # heads of 16: 8 columns a half and whole value rows
    hd = 16
    heads = N // hd - 2
    width = (heads + 2) * hd
    cache = [torch.zeros(2, 1, 16, hd, device=DEV, dtype=torch.bfloat16) for _ in range(4)]
    pos, slots = torch.arange(T, device=DEV, dtype=torch.int32), torch.randperm(32, device=DEV)[:T]
    cs = ref.make_cos_sin_cache(hd, 32).to(DEV)
    own = ops.ProductSums(part[..., :width].contiguous(), sx, sw[:width] if scaled else None)
    q = ops.rope_and_cache(own, heads, pos, cs, *cache[:2], slots)
    q2 = ops.rope_and_cache(y[:, :width].contiguous(), heads, pos, cs, *cache[2:], slots)
    assert torch.equal(cache[1], cache[3])
    for a, b in ((q, q2), (cache[0], cache[2])):
        torch.testing.assert_close(a.float(), b.float(), atol=2.0 ** -20, rtol=2.0 ** -7)
