"""Feed-forward and projection modules at sizes whose products are tiled ones
(csrc/tiled_gemm.h): which form a module hands on, and what its reader makes of it."""
import dataclasses

import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.engine.quant import Fp8Linear, _swap_linears
from kubeai_amd.models.config import PRESETS
from kubeai_amd.models.llama import MLP, MoEMLP

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _module(kind, preset, fp8, **sizes):
    torch.manual_seed(0)
    cfg = dataclasses.replace(PRESETS[preset], **sizes)
    with torch.device(DEV):
        m = kind(cfg).bfloat16().requires_grad_(False)
    if fp8:
        _swap_linears(m)
    return m


class _Down(torch.nn.Module):
    """Keeps the fp8 rows that it is given."""

    def forward_quantized(self, xq, x_scale):
        self.rows = xq, x_scale
        return xq


def _same_fp8(a, b):
    assert torch.equal(a[1], b[1])
    assert torch.equal(a[0].view(torch.uint8), b[0].view(torch.uint8))


@pytest.mark.parametrize("T", [160, 640, 700])
def test_fp8_activation_stays_in_fp32_until_its_conversion(T):
    m = _module(MLP, "llama-tiny", True, hidden_size=2048, intermediate_size=4096)
    m.down_proj = _Down()
    x = ops.quant_fp8(torch.randn(T, 2048, device=DEV, dtype=torch.bfloat16))
    assert ops._tiled_better(T, 8192, 2048, fp8=True)
    m(x)
    _same_fp8(m.down_proj.rows, ops.silu_and_mul_fp8(m.gate_up_proj.forward_quantized(*x)))


def test_fp8_activation_of_experts_stays_in_fp32_until_its_conversion(monkeypatch):
    m = _module(MoEMLP, "mixtral-tiny", True, hidden_size=512, intermediate_size=1024)
    x = torch.randn(300, 512, device=DEV, dtype=torch.bfloat16)
    calls, plain = [], ops.grouped_linear

    def kept(rows, *args, **kw):
        y = plain(rows, *args, **kw)
        calls.append(((rows, kw["scales"][0]), y))
        return y

    monkeypatch.setattr(ops, "grouped_linear", kept)
    with torch.inference_mode():
        m(x)
    (_, h), (a, _) = calls
    assert h.shape == (300 * m.top_k, 2048)
    _same_fp8(a, ops.silu_and_mul_fp8(h))


def _fp8_product(M, N, K):
    torch.manual_seed(M)
    x, w = (torch.randn(n, K, device=DEV).to(torch.float8_e4m3fn) for n in (M, N))
    return x, w, torch.rand(M, device=DEV) + 0.1, torch.rand(N, device=DEV) + 0.1


def _near(y, x, w, sx, sw):
    """bf16 keeps 8 bits (2^-8 of a value); fp32 sums of 2048 terms of up to 2^-13 of
    their magnitudes."""
    a, b = x.double(), w.double()
    s = sx.double().view(-1, 1) * sw.double().view(1, -1)
    want, size = (a @ b.T) * s, (a.abs() @ b.abs().T) * s
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -13 * size).all()


@pytest.mark.parametrize("M,N", [(700, 2048), (32, 49152)])
def test_fp8_scales_of_other_forms_go_to_the_library(M, N):
    """Off a 16-byte boundary, one for all rows and columns, followed by autograd."""
    x, w, sx, sw = _fp8_product(M, N, 2048)
    assert ops._tiled_better(M, N, 2048, fp8=True)
    odd = torch.empty(N + 1, device=DEV)[1:].copy_(sw).view(1, -1)
    assert odd.data_ptr() % 16
    _near(ops.linear_fp8(x, sx, w, odd), x, w, sx, sw)
    one = torch.full((1,), 0.5, device=DEV)
    _near(ops.linear_fp8(x, one, w, one.view(1, 1)), x, w, one, one)
    assert ops.linear_fp8(x, sx.clone().requires_grad_(), w, sw.view(1, -1)).requires_grad
    for refused in (sw, sw.view(-1, 1), sw.double().view(1, -1)):
        with pytest.raises(RuntimeError):
            ops.linear_fp8(x, sx, w, refused)


def test_fp8_results_of_another_shape_go_to_the_library():
    x, w, sx, sw = _fp8_product(700, 2048, 2048)
    assert ops._tiled_better(700, 2048, 2048, fp8=True)
    for rows in (0, 710):
        out = torch.empty(rows, 2048, device=DEV, dtype=torch.bfloat16)
        assert ops.linear_fp8(x, sx, w, sw.view(1, -1), out=out) is out
        assert out.shape == (700, 2048)
        _near(out, x, w, sx, sw)


@pytest.mark.parametrize("M,N,K", [
    (8, 8192, 512),   # (cut along K)
    (12, 16384, 512),
    (1, 65536, 4096),
    (16, 28672, 4096),
    (40, 1024, 16384),  # long rows
])
def test_what_the_streaming_product_does_not_take_goes_to_the_library(M, N, K, monkeypatch):
    """The forms of scales, bias and result that it has no part in give what the
    library gives for them; the usual ones are its own."""
    x, w, sx, sw = _fp8_product(M, N, K)
    assert ops._streams_better(M, N, K, fp8=True)
    calls = []
    own = ops._C.skinny_linear
    monkeypatch.setattr(ops._C, "skinny_linear", lambda *a: calls.append(a) or own(*a))
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    assert ops.linear_fp8(x, sx, w, sw.view(1, -1), out=out) is out
    _near(out, x, w, sx, sw)
    bias = torch.randn(N, device=DEV, dtype=torch.bfloat16)
    got = ops.linear_fp8(x, sx, w, sw.view(1, -1), bias)
    assert len(calls) == 2
    assert ((got.double() - out.double() - bias.double()).abs()
            <= 2.0 ** -7 * (out.double().abs() + bias.double().abs())).all()
    # one scale for all, as the library takes it
    one = torch.full((1,), 0.5, device=DEV)
    _near(ops.linear_fp8(x, one, w, one.view(1, 1)), x, w, one, one)
    # a result of another shape is fitted
    for rows in (0, M + 3):
        other = torch.empty(rows, N, device=DEV, dtype=torch.bfloat16)
        assert ops.linear_fp8(x, sx, w, sw.view(1, -1), out=other) is other
        assert other.shape == (M, N)
        _near(other, x, w, sx, sw)
    # what follows the operation sees it
    assert ops.linear_fp8(x, sx.clone().requires_grad_(), w, sw.view(1, -1)).requires_grad

    class Seen(torch.utils._python_dispatch.TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func._schema.name)
            return func(*args, **(kwargs or {}))

    with Seen() as seen:
        ops.linear_fp8(x, sx, w, sw.view(1, -1))
    assert "aten::_scaled_mm" in seen.names
    assert len(calls) == 2
    with pytest.raises(RuntimeError):
        ops.linear_fp8(x, sx, w, sw.double().view(1, -1))


def test_the_streaming_product_refuses_scales_and_bias_in_host_memory():
    x, w, sx, sw = _fp8_product(8, 64, 512)
    y, bias = (torch.empty(n, 64, device=DEV, dtype=torch.bfloat16) for n in (8, 1))
    ops._C.skinny_linear(y, x, w, sx, sw, bias.zero_())
    _near(y, x, w, sx, sw)
    for args in ((sx.cpu(), sw, bias), (sx, sw.cpu(), bias), (sx, sw, bias.cpu())):
        with pytest.raises(RuntimeError):
            ops._C.skinny_linear(y, x, w, *args)


class _Rows(torch.nn.Module):
    """Keeps the rows that it is given."""

    def forward(self, x):
        self.x = x
        return x


def _spied(monkeypatch, name):
    calls, plain = [], getattr(ops, name)

    def spy(*args, **kw):
        calls.append(plain(*args, **kw))
        return calls[-1]

    monkeypatch.setattr(ops, name, spy)
    return calls


@pytest.mark.parametrize("T", [97, 130, 300])
@pytest.mark.parametrize("gelu", [False, True])
def test_bf16_activation_behind_gate_and_up(T, gelu, monkeypatch):
    """The bounds of test_activations_of_gate_and_up (test_tiled_linear_gpu.py)."""
    m = _module(MLP, "gemma2-tiny" if gelu else "llama-tiny", False, hidden_size=2048,
                intermediate_size=5248)
    assert m.gelu == gelu
    m.down_proj = _Rows()
    x = torch.randn(T, 2048, device=DEV, dtype=torch.bfloat16)
    calls = _spied(monkeypatch, "_tiled_linear")
    with torch.inference_mode():
        m(x)
    assert len(calls) == 1 and calls[0] is m.down_proj.x
    w = m.gate_up_proj.weight.double()
    (g, u), (e, f) = (x.double() @ w.T).chunk(2, -1), (
        2.0 ** -13 * (x.double().abs() @ w.abs().T)).chunk(2, -1)
    fn = torch.nn.functional
    right = (fn.gelu(g, approximate="tanh") if gelu else fn.silu(g)) * u
    tol = 2.0 ** -8 * right.abs() + 1.2 * e * u.abs() + f * (g.abs() + 1.2 * e) + 1e-5
    assert ((m.down_proj.x.double() - right).abs() <= tol).all()


def test_logits_go_through_the_tiled_product(monkeypatch):
    calls = _spied(monkeypatch, "_tiled_linear")
    x = torch.randn(40, 2048, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(98304, 2048, device=DEV, dtype=torch.bfloat16)
    one = torch.ones(1, device=DEV)
    _near(ops.linear(x, w), x, w, one, one)
    x, w, sx, sw = _fp8_product(32, 49152, 2048)
    _near(ops.linear_fp8(x, sx, w, sw.view(1, -1)), x, w, sx, sw)
    assert len(calls) == 2


def _sums(T, N, K, fp8, monkeypatch, rope=False):
    """A module's product as sums of the tiled kernel, checked against 64 bits, and
    the bf16 rows that its reader makes of them."""
    from kubeai_amd.models.llama import EngineLinear

    torch.manual_seed(T)
    lin = EngineLinear(K, N, bias=False, device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(T, K, device=DEV, dtype=torch.bfloat16)
    calls = _spied(monkeypatch, "tiled_sums")
    if fp8:
        lin = Fp8Linear(lin.weight)
        x, sx = ops.quant_fp8(x)
        got, w, sw = lin.sums_quantized(x, sx, rope), lin.weight_fp8, lin.weight_scale
    else:
        got, w = lin.sums(x, rope), lin.weight
        sx = sw = torch.ones(1, device=DEV)
    assert len(calls) == 1 and calls[0] is got and got.part.shape[0] > 1
    y = torch.zeros(T, N, device=DEV)
    for part in got.part:  # in this order, in fp32
        y += part
    if fp8:
        y = y * sx[:, None] * sw.view(1, -1)
    _near(y, x, w, sx, sw)
    return got, y.bfloat16()


@pytest.mark.parametrize("T", [40, 97, 128, 300])
@pytest.mark.parametrize("fp8", [False, True])
def test_norms_of_tiled_sums(T, fp8, monkeypatch):
    """As the norms of the rows that the sums make; the two may contract their fp32
    products either way, which moves one output in some hundreds by one step of its
    type, and a scale by its last bit."""

    def near(a, b, step):
        a, b = a.float(), b.float()
        assert (a != b).sum().item() <= 2 + a.numel() // 100
        torch.testing.assert_close(a, b, atol=1e-6, rtol=step)

    got, y = _sums(T, 2048, 8192, fp8, monkeypatch)
    r, w1, w2 = (torch.randn(n, 2048, device=DEV, dtype=torch.bfloat16).squeeze(0)
                 for n in (T, 1, 1))
    near(ops.rmsnorm(got, w1, 1e-5), ops.rmsnorm(y, w1, 1e-5), 2.0 ** -7)
    r1, r2 = r.clone(), r.clone()
    (a, _), (b, _) = (ops.fused_add_rmsnorm(got, r1, w1, 1e-5),
                      ops.fused_add_rmsnorm(y.clone(), r2, w1, 1e-5))
    assert torch.equal(r1, r2)
    near(a, b, 2.0 ** -7)
    for (a, sa), (b, sb) in (
        (ops.rmsnorm_fp8(got, w1, 1e-5), ops.rmsnorm_fp8(y, w1, 1e-5)),
        (ops.fused_add_rmsnorm_fp8(got, r1, w1, 1e-5), ops.fused_add_rmsnorm_fp8(y, r2, w1, 1e-5)),
    ):
        near(a, b, 2.0 ** -3)
        torch.testing.assert_close(sa, sb, atol=0, rtol=1e-6)
    assert torch.equal(r1, r2)
    for a, b in zip(*(ops.add_and_norm(ops.BranchNorm(x, w1, 1e-5), r, w2, 1e-5)
                      for x in (got, y))):
        assert torch.equal(a, b)


def test_scales_that_autograd_follows_keep_the_whole_product():
    lin = Fp8Linear(torch.randn(2048, 8192, device=DEV, dtype=torch.bfloat16))
    x, sx = ops.quant_fp8(torch.randn(300, 8192, device=DEV, dtype=torch.bfloat16))
    assert isinstance(lin.sums_quantized(x, sx), ops.ProductSums)
    assert lin.sums_quantized(x, sx.requires_grad_()) is None


@pytest.mark.parametrize("T", [40, 97, 128])
@pytest.mark.parametrize("fp8", [False, True])
def test_rotation_of_tiled_sums(T, fp8, monkeypatch):
    n_q, n_kv, hd = 24, 4, 64
    got, y = _sums(T, (n_q + 2 * n_kv) * hd, 12288, fp8, monkeypatch, rope=True)
    pos = torch.randint(0, 900, (T,), device=DEV, dtype=torch.int32)
    slots = torch.randperm(320, device=DEV)[:T]
    slots[2] = -1
    cos_sin = torch.randn(1000, hd, device=DEV)
    caches = [torch.zeros(20, n_kv, 16, hd, device=DEV, dtype=torch.bfloat16) for _ in range(4)]
    a = ops.rope_and_cache(got, n_q, pos, cos_sin, *caches[:2], slots)
    b = ops.rope_and_cache(y, n_q, pos, cos_sin, *caches[2:], slots)
    assert torch.equal(a, b)
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
