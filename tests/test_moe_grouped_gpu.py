"""Device-side routing and grouped expert products at the edges of their tiles
(16-row tiles, 64 columns a workgroup, 128/256-byte steps of K, several passes
for an expert with many rows) and skinny products at theirs.

The reference rounds where the kernels do (each product and the activation to
bf16), so what is left is fp32 sums in another order, which moves a rounded
intermediate by one bf16 step (2^-8) now and then: bounded as 2^-7 of the
largest value of a row, and 1e-3 in the norm."""
import pytest
import torch
import torch.nn.functional as F

import kubeai_amd.ops as ops
from kubeai_amd.engine.quant import Fp8Linear
from kubeai_amd.models.config import PRESETS, ModelArchConfig
from kubeai_amd.models.llama import MoEMLP

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _close(got, want):
    got, want = got.float(), want.float()
    assert (got - want).norm() <= 2e-3 * want.norm() + 1e-6
    big = want.abs().amax(-1, keepdim=True)
    assert ((got - want).abs() <= 2.0 ** -7 * big + 1e-6).all()


def _mm(x, w):
    return (x.double() @ w.double().T).float()


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 64, 65, 96])
@pytest.mark.parametrize("N,K", [(4, 32), (60, 64), (64, 96), (100, 544), (4100, 1312),
                                 (16640, 256)])
def test_skinny_linear(M, N, K):
    from kubeai_amd import _C

    torch.manual_seed(M + N + K)
    wide = torch.randn(M, K + 16, device=DEV, dtype=torch.bfloat16)
    x, w = wide[:, :K], torch.randn(N, K, device=DEV, dtype=torch.bfloat16)
    y = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    b = torch.randn(N, device=DEV, dtype=torch.bfloat16)
    _C.skinny_linear(y, x, w, None, None, None)
    _close(y, _mm(x, w))
    _C.skinny_linear(y, x, w, None, None, b)
    _close(y, _mm(x, w) + b.float())
    if K % 64:
        return
    x8, w8 = x.contiguous().to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
    sx, sw = torch.rand(M, device=DEV) + 0.1, torch.rand(N, device=DEV) + 0.1
    _C.skinny_linear(y, x8, w8, sx, sw, b)
    _close(y, _mm(x8.float(), w8.float()) * sx[:, None] * sw + b.float())


@pytest.mark.parametrize("M,N,K", [(1, 6144, 4096), (33, 4096, 4096), (7, 4096, 14336),
                                   (64, 4096, 14336), (16, 128256, 4096)])
def test_skinny_linear_large(M, N, K):
    from kubeai_amd import _C

    torch.manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(N, K, device=DEV, dtype=torch.bfloat16)
    y = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    _C.skinny_linear(y, x, w, None, None, None)
    _close(y, _mm(x, w))


def _experts(E, I, H):
    gu = torch.randn(E, 2 * I, H, device=DEV, dtype=torch.bfloat16) * H ** -0.5
    dn = torch.randn(E, H, I, device=DEV, dtype=torch.bfloat16) * I ** -0.5
    return gu, dn


@pytest.mark.parametrize("T,E,top", [(1, 8, 2), (3, 1, 1), (17, 5, 3), (40, 8, 2), (97, 32, 8),
                                     (300, 4, 2)])
@pytest.mark.parametrize("one_expert", [False, True])
def test_moe(T, E, top, one_expert):
    torch.manual_seed(T * E)
    H, I = 256, 160
    x = torch.randn(T, H, device=DEV, dtype=torch.bfloat16)
    router = torch.randn(E, H, device=DEV, dtype=torch.bfloat16)
    if one_expert:  # every token's first choice is the last expert
        x[:, 0] = 100.0
        router[:, 0] = 0.0
        router[E - 1, 0] = 5.0
    gu, dn = _experts(E, I, H)
    got = ops.moe_mlp(x, router, top, gu, dn)
    z = _mm(x, router)
    v, idx = z.topk(top, -1)
    w = torch.softmax(v, -1)
    want = torch.zeros(T, H, device=DEV)
    for e in range(E):
        h = _mm(x, gu[e]).bfloat16().float()
        g, u = h.chunk(2, -1)
        a = (F.silu(g) * u).bfloat16()
        y = _mm(a, dn[e]).bfloat16().float()
        want += (w * (idx == e)).sum(-1, keepdim=True) * y
    _close(got, want)


def test_module_routes():
    """fp8 and bf16 modules against their per-expert route, weights copied in
    after construction, and a module whose tensor has left the stack."""
    cfg = ModelArchConfig(architecture="mixtral", hidden_size=256, intermediate_size=192,
                          num_local_experts=4, num_experts_per_tok=2)
    torch.manual_seed(5)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            m = MoEMLP(cfg)
    finally:
        torch.set_default_dtype(prev)
    x = torch.randn(37, 256, device=DEV, dtype=torch.bfloat16)

    def both():
        grouped = m._grouped(x)
        assert grouped is not None
        m._on_device = lambda x: False
        one_by_one = m(x)
        del m._on_device
        # the per-expert route rounds weights and partial sums to bf16
        assert (grouped - one_by_one).float().norm() < 0.02 * one_by_one.float().norm()
        _close(m._sorted(x), grouped)  # the same roundings, library products
        return grouped

    with torch.inference_mode():
        both()
        for e in m.experts:
            e.down_proj.weight.copy_(torch.randn_like(e.down_proj.weight))
        both()
        for e in m.experts:
            e.gate_up_proj = Fp8Linear(e.gate_up_proj.weight)
            e.down_proj = Fp8Linear(e.down_proj.weight)
        assert m._grouped(x) is None  # the modules' tensors are not the stack's
        m.stack_experts()
        both()
        m.experts[1].down_proj.weight_fp8 = m.experts[1].down_proj.weight_fp8.clone()
        assert m._grouped(x) is None
        big = torch.randn(700, 256, device=DEV, dtype=torch.bfloat16)
        many, few = m(big)[:37].float(), m(big[:37].contiguous()).float()
        assert (many - few).norm() < 0.02 * few.norm()  # sorted, and per expert
    assert PRESETS["mixtral-8x7b"].num_local_experts <= 32


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("I", [192, 256])
def test_which_product(fp8, I):
    """The tiled product from 161 (fp8) or 225 tokens on where it takes rows of
    both widths, with the streaming one's results, also from a graph."""
    cfg = ModelArchConfig(architecture="mixtral", hidden_size=256, intermediate_size=I,
                          num_local_experts=8, num_experts_per_tok=2)
    torch.manual_seed(I)
    with torch.device(DEV):
        m = MoEMLP(cfg).bfloat16()
    if fp8:
        for e in m.experts:
            e.gate_up_proj = Fp8Linear(e.gate_up_proj.weight)
            e.down_proj = Fp8Linear(e.down_proj.weight)
    m.stack_experts()
    calls = []
    ordered = m._sorted
    m._sorted = lambda x: calls.append(x.shape[0]) or ordered(x)
    takes = not fp8 or I % 128 == 0
    with torch.inference_mode():
        for T in (160, 161, 224, 225, 256, 257):
            x = torch.randn(T, 256, device=DEV, dtype=torch.bfloat16)
            got = m(x)
            tiled = T > 256 or takes and T > (160 if fp8 else 224)
            assert calls == ([T] if tiled else [])
            calls.clear()
            if T > m.GROUPED_MAX_TOKENS:
                continue
            want = m._grouped(x)
            if fp8:
                # an activation row whose largest value lands one bf16 step away
                # is scaled, and rounded, anew: by up to 2^-4 of each value
                assert (got - want).float().norm() < 2.0 ** -5 * want.float().norm()
            else:
                _close(got, want)
        x = torch.randn(256, 256, device=DEV, dtype=torch.bfloat16)
        m(x)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = m(x)
        for _ in range(3):
            x.copy_(torch.randn_like(x))
            x[: 128] = x[0]  # other row counts than the recorded step's
            g.replay()
            assert torch.equal(out, m(x))


def test_rows_that_begin_anywhere():
    """Hidden rows that are not on a 16-byte boundary take the per-expert route."""
    cfg = ModelArchConfig(architecture="mixtral", hidden_size=128, intermediate_size=64,
                          num_local_experts=4, num_experts_per_tok=2)
    with torch.device(DEV):
        m = MoEMLP(cfg).bfloat16()
    m.stack_experts()
    for T in (5, 300):
        odd = torch.randn(T * 128 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(T, 128)
        with torch.inference_mode():
            got, want = m(odd).float(), m(odd.clone()).float()
        # the per-expert route rounds weights and partial sums to bf16
        assert (got - want).norm() < 0.02 * want.norm()


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("E,top", [(4, 2), (5, 5), (32, 8), (1, 1)])
def test_scores_that_are_not_finite(bad, E, top):
    """The same weights as topk and softmax give, NaN among them, and every
    token's experts differ and are in range."""
    torch.manual_seed(E)
    x = torch.randn(9, 64, device=DEV, dtype=torch.bfloat16)
    router = torch.randn(E, 64, device=DEV, dtype=torch.bfloat16)
    x[0, 3] = x[4, 7] = bad
    x[6, :] = bad
    router[E // 2, 5] = bad  # an infinite or NaN score of every other token
    x[8] = 0.0  # (0 times infinity)
    z = x.float() @ router.float().T
    v = z.topk(top, -1).values
    want = torch.softmax(v, -1)
    weight, begin, src, place = ops.moe_route(x, router, top)
    torch.testing.assert_close(weight, want, atol=1e-5, rtol=1e-4, equal_nan=True)
    b, s, p = begin.tolist(), src.tolist(), place.tolist()
    assert b[0] == 0 and b[-1] == 9 * top and sorted(p) == list(range(9 * top))
    for e in range(E):  # a token is at an expert once
        rows = s[b[e] : b[e + 1]]
        assert rows == sorted(set(rows))


def test_a_router_that_is_not_finite_reaches_the_output():
    cfg = ModelArchConfig(architecture="mixtral", hidden_size=128, intermediate_size=64,
                          num_local_experts=4, num_experts_per_tok=2)
    with torch.device(DEV):
        m = MoEMLP(cfg).bfloat16()
    m.stack_experts()
    with torch.inference_mode():
        m.gate.weight[2, 0] = float("nan")
        for T in (5, 300):
            x = torch.randn(T, 128, device=DEV, dtype=torch.bfloat16)
            assert m._grouped(x) is not None or T > m.GROUPED_MAX_TOKENS
            assert m(x).isnan().all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("gathered", [False, True])
def test_experts_over_more_than_2_gib_of_rows(fp8, gathered):
    rows, N, K = 270_000, 64, 8192 if fp8 else 4096
    torch.manual_seed(3)
    x = torch.empty(rows, K, device=DEV, dtype=torch.bfloat16).normal_()
    w = torch.randn(2, N, K, device=DEV, dtype=torch.bfloat16)
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(rows, device=DEV) + 0.5, torch.rand(2, N, device=DEV) + 0.5
    if gathered:
        src = torch.tensor([rows - 1, 0, 5, rows - 2, 131_072] * 30, device=DEV, dtype=torch.int32)
        begin, at = (0, 70, 150), src.long()
    else:
        src, begin, at = None, (0, 97, rows), torch.arange(rows, device=DEV)
    y = torch.empty(begin[-1], N, device=DEV, dtype=torch.bfloat16)
    ops._C.skinny_experts(y, x, w, sx, sw,
                          torch.tensor(begin, dtype=torch.int32, device=DEV), src)
    for e in range(2):
        lo, hi = begin[e], begin[e + 1]
        for part in (slice(lo, min(lo + 200, hi)), slice(max(lo, hi - 200), hi)):
            a, b = x[at[part]].double(), w[e].double()
            s = sx[at[part], None].double() * sw[e].double() if fp8 else 1.0
            want, size = (a @ b.T) * s, (a.abs() @ b.abs().T) * s
            # one rounding to bf16; fp32 sums
            assert ((y[part].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * size).all()


@pytest.mark.parametrize("E,R,N", [(1, 3, 20), (5, 4, 100), (8, 24, 28672), (64, 9, 68),
                                   (65, 200, 36), (130, 40, 260), (130, 1, 16), (8, 300, 132)])
@pytest.mark.parametrize("fp8", [False, True])
def test_experts_without_rows(E, R, N, fp8):
    """Whichever experts have rows, two waves a workgroup and four, more experts than a
    wave has lanes; rows behind the last expert's stay as they are."""
    K = 192
    torch.manual_seed(E + R)
    w = torch.randn(E, N, K, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(R + 2, K, device=DEV, dtype=torch.bfloat16)
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(R + 2, device=DEV) + 0.5, torch.rand(E, N, device=DEV) + 0.5
    for own in (range(E), [0], [E - 1], [E // 2, E - 1], [i for i in (0, 63, 64) if i < E]):
        own = list(own)
        counts = torch.bincount(
            torch.tensor(own)[torch.randint(len(own), (R,))], minlength=E)
        begin = [0] + counts.cumsum(0).tolist()
        y = torch.full((R + 2, N), 7.0, device=DEV, dtype=torch.bfloat16)
        ops._C.skinny_experts(y, x, w, sx, sw,
                              torch.tensor(begin, dtype=torch.int32, device=DEV), None)
        assert (y[R:] == 7).all()
        for e in range(E):
            rows = slice(begin[e], begin[e + 1])
            a, b = x[rows].double(), w[e].double()
            s = sx[rows, None].double() * sw[e].double() if fp8 else 1.0
            want, size = (a @ b.T) * s, (a.abs() @ b.abs().T) * s
            # one rounding to bf16; fp32 sums
            assert ((y[rows].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * size).all()


@pytest.mark.parametrize("R,N", [(69, 68), (132, 68), (133, 68), (300, 68), (69, 9000),
                                 (133, 9000)])
@pytest.mark.parametrize("K", [64, 128, 192, 320, 448, 1088])
@pytest.mark.parametrize("fp8", [False, True])
def test_experts_of_many_rows(R, N, K, fp8):
    """64 and 96 rows a pass, steps of 128 and 256 bytes: one to more than are under way,
    whole ones and not; several passes (all rows of one expert), gathered rows; four waves a
    workgroup and eight (bf16 of 9000 columns)."""
    E = 3
    torch.manual_seed(R + K)
    w = torch.randn(E, N, K, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(R, K, device=DEV, dtype=torch.bfloat16)
    src = torch.randint(R, (R,), device=DEV, dtype=torch.int32)
    sx = sw = None
    if fp8:
        x, w = x.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn)
        sx, sw = torch.rand(R, device=DEV) + 0.5, torch.rand(E, N, device=DEV) + 0.5
    for begin in ([0, R // 3, R // 3 + 1, R], [0, 0, R, R]):
        for rows in (None, src):
            y = torch.empty(R, N, device=DEV, dtype=torch.bfloat16)
            ops._C.skinny_experts(y, x, w, sx, sw,
                                  torch.tensor(begin, dtype=torch.int32, device=DEV), rows)
            at = torch.arange(R, device=DEV) if rows is None else rows.long()
            for e in range(E):
                part = slice(begin[e], begin[e + 1])
                a, b = x[at[part]].double(), w[e].double()
                s = sx[at[part], None].double() * sw[e].double() if fp8 else 1.0
                want, size = (a @ b.T) * s, (a.abs() @ b.abs().T) * s
                # one rounding to bf16; fp32 sums
                off = (y[part].double() - want).abs()
                assert (off <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * size).all()
