"""All experts' products of a large step in one launch, at the edges of its
tiles (128, 192 or 256 rows, 256 columns, 128 bytes of K): empty experts, one row,
one more than a tile, more experts than a wave has lanes, strided weights and
gathered rows, and what it leaves to the library.

Against the product in 64 bits: rounding to the 8 significant bits of bf16
moves a result by at most half of 2^-7 of itself, fp32 sums of K terms by at most K 2^-24 of the sum of the
terms' sizes (K <= 1024: 2^-14)."""
import pytest
import torch

import kubeai_amd.ops as ops
from kubeai_amd.models.mixers import RoutedGatedMoE, RoutedSquaredReluMoE

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _reference(x, w, counts, src):
    rows = x.double()[src.long()]
    y, size = [], []
    for e, part in enumerate(rows.split(counts)):
        y.append(part @ w[e].double().T)
        size.append(part.abs() @ w[e].double().abs().T)
    return torch.cat(y), torch.cat(size)


@pytest.mark.parametrize("counts,N,K", [
    ([1], 4, 64),
    ([0, 127, 0, 128, 129, 0], 260, 128),
    ([255, 1, 257, 300], 252, 192),
    ([3000, 0, 17], 1028, 1024),
    ([5] * 70 + [140], 64, 64),
    ([2000] * 8, 2048, 64),
    ([255, 0, 257, 1, 1500], 7172, 256),  # tiles of 192 rows
    ([191, 0, 193, 1, 2600], 4100, 320),  # of 256
])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("offsets", [False, True])
def test_grouped_linear(counts, N, K, fp8, offsets):
    torch.manual_seed(sum(counts) + N)
    E, R, dt = len(counts), sum(counts), torch.bfloat16
    K = K * 2 if fp8 else K
    x = torch.randn(R // 2 + 1, K + 32, device=DEV, dtype=dt)[:, :K]
    wide = torch.randn(N, E * K + 64, device=DEV, dtype=dt)  # experts side by side
    src = torch.randint(0, x.shape[0], (R,), device=DEV, dtype=torch.int32)
    sx, sw = torch.rand(x.shape[0], device=DEV) + 0.1, torch.rand(E, N, device=DEV) + 0.1
    if fp8:
        x = x.contiguous().to(torch.float8_e4m3fn)
        wide = wide.to(torch.float8_e4m3fn)
    w = wide[:, : E * K].unflatten(1, (E, K)).transpose(0, 1)
    c = torch.tensor(counts, device=DEV, dtype=torch.int32)
    bounds = torch.nn.functional.pad(c.cumsum(0, dtype=torch.int32), (1, 0)) if offsets else c
    assert ops.grouped_linear_takes(x, w)
    want, size = _reference(x, w, counts, src)
    tol = 2.0 ** -8 * want.abs() + 2.0 ** -14 * size
    if fp8:
        s = sx[src.long(), None].double() * torch.repeat_interleave(sw, c, 0).double()
        got = ops.grouped_linear(x, w, bounds, src=src, scales=(sx, sw))
        # two more fp32 products per result
        assert ((got.double() - want * s).abs() <= tol * s * (1 + 2.0 ** -8) + 1e-30).all()
        return
    got = ops.grouped_linear(x, w, bounds, src=src)
    assert ((got.double() - want).abs() <= tol + 1e-30).all()
    rows = x.index_select(0, src)
    assert torch.equal(ops.grouped_linear(rows, w, bounds), got)
    rw = torch.rand(R, 1, device=DEV)
    r = got.float().clamp(min=0)
    sq = ops.grouped_linear(rows, w, bounds, square=rw)
    assert torch.equal(sq, (r * r * rw).to(dt))


@pytest.mark.parametrize("kind", [RoutedSquaredReluMoE, RoutedGatedMoE])
@pytest.mark.parametrize("ff", [128, 96])  # 96: not a whole number of steps of K
def test_module_routes(kind, ff):
    """The module's large step against its own small ones (every expert, dense)."""
    torch.manual_seed(ff)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            m = kind(256, 8, 2, ff, shared_ff=64)
    finally:
        torch.set_default_dtype(prev)
    x = torch.randn(700, 256, device=DEV, dtype=torch.bfloat16)
    with torch.inference_mode():
        many = m(x).float()
        few = torch.cat([m(p.contiguous()) for p in x.split(200)]).float()
    # the dense step rounds the weighted activation where this one rounds the
    # expert's output: both by up to 2^-8 of their terms
    assert (many - few).norm() <= 1e-2 * few.norm()
