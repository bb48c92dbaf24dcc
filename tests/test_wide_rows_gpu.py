"""Per-head maps and the query/key norm with half rotation in whole units, at the
edges of their tiles, against float64; sizes beside them take the general kernels."""
import pytest
import torch

from kubeai_amd.ops import seq as sops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("A,B", [(32, 32), (64, 96), (128, 128), (256, 64), (512, 32), (96, 32),
                                 (128, 48)])
@pytest.mark.parametrize("T,H", [(1, 2), (17, 3), (129, 2), (1000, 40)])
@pytest.mark.parametrize("gated", [None, "channel", "head"])
def test_head_linear(T, H, A, B, gated):
    """One rounding to bf16 (2^-9 of the result); fp32 sums of at most 512 terms
    (2^-15 of the magnitudes); the gate's factor is below 1 and within 2^-20."""
    torch.manual_seed(T + A + B)
    wide = torch.randn(T, H, A + 8, device=DEV, dtype=torch.bfloat16)
    x = wide[..., 8:]
    w = torch.randn(H, B, A, device=DEV, dtype=torch.bfloat16)
    gate = {None: None, "channel": torch.randn(T, H * B, device=DEV, dtype=torch.bfloat16),
            "head": torch.randn(T, H, device=DEV, dtype=torch.bfloat16)}[gated]
    out = torch.full((T + 1, H, B + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    sops.head_linear(x, w, gate, out=out[:T, :, 8:])
    xd, wd = x.double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()
    want = torch.bmm(xd, wd).transpose(0, 1)
    size = torch.bmm(xd.abs(), wd.abs()).transpose(0, 1)
    if gate is not None:
        want = want * torch.sigmoid(gate.double()).view(T, H, -1)
    got = out[:T, :, 8:].double()
    assert ((got - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -15).all()
    assert (out[T] == 7).all() and (out[..., :8] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv,half", [(16, 4, 128, 128, 64), (16, 2, 64, 32, 16),
                                           (1, 1, 8, 8, 0), (40, 8, 128, 64, 64),
                                           (96, 8, 128, 128, 32), (3, 1, 24, 24, 12),
                                           (200, 8, 128, 8, 64)])
@pytest.mark.parametrize("normed", [True, False])
def test_qknorm_rope_half(dtype, H, G, D, Dv, half, normed):
    """fp32 throughout and one rounding to the type; the sums of squares over at
    most 25600 values and the turn by fp32 angles up to 4000 (2^-24 of them each for
    the position's product and its use: 2^-11 of the pair's size)."""
    torch.manual_seed(H + D)
    T, bs, blocks = 5, 16, 4
    qkv = torch.randn(T, (H + G) * D + G * Dv, device=DEV).to(dtype)
    q, k, v = qkv.split([H * D, G * D, G * Dv], dim=-1)
    q, k, v = q.unflatten(-1, (H, D)), k.unflatten(-1, (G, D)), v.unflatten(-1, (G, Dv))
    qw = torch.rand(H * D, device=DEV) + 0.5 if normed else None
    kw = torch.rand(G * D, device=DEV) + 0.5 if normed else None
    pos = torch.tensor([0, 1, 77, 2048, 4000], dtype=torch.int32, device=DEV)
    inv = 10000.0 ** (-torch.arange(half, device=DEV, dtype=torch.float32) / max(half, 1))
    slots = torch.tensor([3, 40, -1, 17, 63], device=DEV)
    kc = torch.zeros(blocks, G, bs, D, device=DEV, dtype=dtype)
    vc = torch.zeros(blocks, G, bs, Dv, device=DEV, dtype=dtype)

    def want(x, w):
        y = x.double()
        if w is not None:
            y = y.flatten(1)
            y = y / (y.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()
            y = y.view(x.shape)
        angle = (pos.float()[:, None] * inv).double()[:, None]
        a, b = y[..., :half], y[..., half : 2 * half]
        pair = (a * a + b * b).sqrt()
        turned = torch.cat([a * angle.cos() - b * angle.sin(),
                            b * angle.cos() + a * angle.sin(), y[..., 2 * half :]], -1)
        return turned, torch.cat([pair, pair, y[..., 2 * half :].abs()], -1)

    (wq, sq), (wk, sk) = want(q, qw), want(k, kw)
    v_was = v.clone()
    sops.qknorm_rope_half_and_cache(q, k, v, qw, kw, 1e-5, pos, inv, kc, vc, slots)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((q.double() - wq).abs() <= rel * wq.abs() + 2.0 ** -11 * sq + 1e-6).all()
    kept = 0
    for t, s in enumerate(slots.tolist()):
        if s < 0:
            continue
        kept += 1
        ck, cv = kc[s // bs, :, s % bs].double(), vc[s // bs, :, s % bs]
        assert ((ck - wk[t]).abs() <= rel * wk[t].abs() + 2.0 ** -11 * sk[t] + 1e-6).all()
        assert torch.equal(cv, v_was[t])
    written = kc.flatten(1, 1).transpose(1, 2).reshape(blocks * bs, -1)
    assert (written.abs().sum(-1) > 0).sum() == kept
