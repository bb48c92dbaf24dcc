"""Post-norm + residual + pre-norm at the edges of its register forms (1024, 2048
and 4096 columns) and beyond them.

Against 64 bits. fp32: the sum of squares of C positive terms is off by at most
C 2^-24 of itself, in practice far less; 2^-20 of the largest value covers its
root and the four roundings after it. bf16 out: half of 2^-7 of the value more."""
import pytest
import torch

from kubeai_amd.ops import seq as sops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("C", [1, 255, 1024, 1025, 2047, 2048, 2049, 4096, 4097, 8200])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["none", "same", "fp32"])
def test_sandwich_norm_rows(C, dtype, kind):
    g = torch.Generator(device=DEV).manual_seed(C)

    def rnd(*s):
        return torch.randn(*s, generator=g, device=DEV)

    x, wa, wb = rnd(5, C), 1 + 0.1 * rnd(C), 1 + 0.1 * rnd(C)
    y = None
    if kind != "none":
        y = rnd(5, C).to(torch.float32 if kind == "fp32" else dtype)
    want = x.double()
    if y is not None:
        b = y.double()
        want = want + b * torch.rsqrt((b * b).mean(-1, keepdim=True) + 1e-5) * wb.double()
    normed = want * torch.rsqrt((want * want).mean(-1, keepdim=True) + 1e-5) * wa.double()
    h = sops.sandwich_rmsnorm(y, wb, x, wa, 1e-5, dtype)
    assert h.dtype == dtype
    assert ((x.double() - want).abs() <= 2.0 ** -20 * want.abs().max()).all()
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((h.double() - normed).abs() <= half * normed.abs()
            + 2.0 ** -20 * normed.abs().max()).all()
