"""Masked attention of prompt portions in bf16, at the edges of its tiles of keys and
queries: runs that end at and beside 16, 32 and 64 keys, portions that continue, windows
and chunks that begin inside 16 keys, cache blocks of 8 to 32, sizes with kernels of
their own and others. Cached rows that no query may see hold NaN, in hidden blocks and
beside visible rows: none reaches a result."""
import pytest
import torch

from kubeai_amd.ops import seq as sops

pytestmark = pytest.mark.gpu

MASKS = [dict(), dict(window=37), dict(window=37, keep_first=20), dict(chunk=40, softcap=5.0)]


@pytest.mark.parametrize("H,G,D,Dv,tied", [
    (6, 1, 128, 128, True), (4, 2, 128, 128, False), (3, 1, 64, 64, True),
    (4, 4, 64, 64, False), (4, 2, 64, 128, False), (5, 1, 192, 128, True),
    (4, 1, 48, 48, False), (2, 1, 128, 256, False), (2, 1, 256, 256, False),
    (2, 2, 256, 240, False), (2, 1, 256, 256, True),
    (2, 1, 256, 224, False)])  # (more than 64 KB of LDS)
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("short", [True, False])
@pytest.mark.parametrize("mask", range(len(MASKS)))
def test_prompt_tiles(H, G, D, Dv, tied, bs, short, mask):
    torch.manual_seed(5)
    opts = dict(MASKS[mask])
    runs = ([(1, 0), (16, 0), (17, 0), (32, 0), (9, 70)] if short else
            [(1, 130), (64, 0), (65, 0), (33, 96), (257, 3), (15, 64)])  # length, first position
    need = [(p + n + bs - 1) // bs for n, p in runs]
    free = (torch.randperm(sum(need)) + 1).tolist()
    tables = torch.zeros(len(runs), max(need), dtype=torch.int32)
    kc = torch.full((sum(need) + 1, G, bs, D), float("nan"), dtype=torch.bfloat16)
    vc = torch.full((sum(need) + 1, G, bs, Dv), float("nan"), dtype=torch.bfloat16)
    for i, (n, p) in enumerate(runs):
        low = max(0, p - opts.get("window", p + 1) + 1, p // opts.get("chunk", p + 1)
                  * opts.get("chunk", 0))
        for b in range(need[i]):
            if (b + 1) * bs <= low and b * bs >= opts.get("keep_first", 0):
                free.pop()  # hidden from the whole portion: block 0, NaN throughout
                continue
            tables[i, b] = at = free.pop()
            seen = min(bs, p + n - b * bs)
            kc[at, :, :seen] = torch.randn(G, seen, D).bfloat16()
            vc[at, :, :seen] = torch.randn(G, seen, Dv).bfloat16()
            gone = [j % bs for j in range(b * bs, min((b + 1) * bs, low))
                    if j >= opts.get("keep_first", 0)]
            kc[at, :, gone] = vc[at, :, gone] = float("nan")
    if tied:
        vc = kc[..., :Dv]
    q = torch.randn(sum(n for n, _ in runs), H, D).bfloat16()
    pos = torch.cat([torch.arange(p, p + n) for n, p in runs]).int()
    if mask % 2:
        opts["slopes"] = torch.rand(H) * 0.1
    if tied:
        opts["key_scale"] = (torch.rand(kc.shape[0], bs, 1) + 0.5).float()

    def run(dev, values, cut):
        meta = sops.SeqMeta.build([(n, 0) for n, _ in runs], pos.to(dev), dev,
                                  block_tables=tables.to(dev))
        k = kc.to(dev)
        v = k[..., :Dv] if values is None else values.to(dev)
        out = torch.zeros(q.shape[0], H, Dv, dtype=cut, device=dev)
        on = {n: x.to(dev) if torch.is_tensor(x) else x for n, x in opts.items()}
        return sops.masked_paged_attention(q.to(dev), k, v, meta, D ** -0.5, out, **on).cpu().float()

    got = run("cuda", None if tied else vc, torch.bfloat16)
    want = run("cpu", vc, torch.float32)
    # A probability and the result are rounded to bf16, each by up to 2^-8 of itself
    # (8 bits, to the nearest): together 2^-7 of the sum of p |v|. The rest is in 32 bits.
    room = run("cpu", vc.abs(), torch.float32) * 2 ** -7 * 1.02 + 1e-5
    assert torch.isfinite(got).all()
    worst = ((got - want).abs() / room).max().item()
    assert worst <= 1, worst
