"""The rows of a large step's experts with the shared expert among them."""
import pytest
import torch

from kubeai_amd import ops
from kubeai_amd.models.mixers import RoutedSquaredReluMoE
from kubeai_amd.ops import seq as sops

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (7, 3, 2), (257, 8, 2), (1025, 5, 3),
                                     (2048, 70, 1), (4096, 8, 2), (4097, 8, 2), (16385, 3, 1)])
def test_one_more_expert_has_every_token(device, T, E, top):
    """The same rows, places and counts as when each token chooses it itself."""
    g = torch.Generator().manual_seed(T)
    idx = torch.rand(T, E, generator=g).argsort(1)[:, :top].int()
    w = torch.rand(T, top, generator=g)
    got = sops.expert_order(idx.to(device), w.to(device), E, every=True)
    more = torch.cat([idx, torch.full((T, 1), E, dtype=torch.int32)], 1)
    want = sops.expert_order(more, torch.cat([w, torch.ones(T, 1)], 1), E + 1)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a.cpu(), b)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [257, 300, 1024, 3000])
@pytest.mark.parametrize("W,E,top,ff,shared", [(256, 4, 2, 128, 128), (512, 8, 2, 448, 448),
                                               (256, 4, 1, 128, 64), (256, 3, 2, 80, 80)])
def test_mixture_with_a_shared_expert(T, W, E, top, ff, shared):
    """Shared experts of the others' size, of another one, and of rows that the tiled
    product does not take, against fp32."""
    torch.manual_seed(T)
    moe = RoutedSquaredReluMoE(W, E, top, ff, shared).to("cuda", torch.bfloat16)
    moe.router.data = moe.router.data.float()
    h = torch.randn(T, W, device="cuda").bfloat16()
    got = moe(h).float()
    up, down, x = moe.up.weight.float(), moe.down.weight.float(), h.float()
    dense, _, _ = sops.router_topk(x @ moe.router.t(), top)
    a = torch.relu(x @ up.t()).square()
    a[:, : E * ff] *= dense.repeat_interleave(ff, 1)
    want = a @ down.t()
    # three roundings to bf16 in a row (2^-9 each, at most), of independent signs
    assert (got - want).norm() / want.norm() < 5e-3
    assert ops.have_hip_ext()


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("T,C,top", [(1, 8, 1), (3, 1000, 2), (70, 1024, 3), (257, 2048, 3),
                                     (5, 2052, 4), (9, 4096, 5), (4, 4100, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norms_of_rows_not_yet_added(device, T, C, top, dtype):
    """The bits of the sum as a launch of its own: rows in registers and longer ones, as
    many choices as are asked for at a time and more."""
    g = torch.Generator().manual_seed(C + top)
    y = torch.randn(T * top, C, generator=g).to(device, dtype)
    place = torch.randperm(T * top, generator=g).int().view(T, top).to(device)
    res = torch.randn(T, C, generator=g).to(device)
    w = [torch.rand(C, generator=g).to(device) + 0.5 for _ in range(2)]
    one, two = res.clone(), res.clone()
    want = sops.sandwich_rmsnorm(sops.combine_expert_rows(y, place), w[0], one, w[1], 1e-5, dtype)
    got = sops.sandwich_rmsnorm(sops.ExpertSum(y, place), w[0], two, w[1], 1e-5, dtype)
    assert torch.equal(got, want) and torch.equal(one, two)


@pytest.mark.gpu
@pytest.mark.parametrize("E,shared,together", [(15, 128, True), (16, 128, False), (4, 64, False)])
def test_where_the_shared_expert_is_among_the_others(monkeypatch, E, shared, together):
    seen, real = [], sops.expert_order

    def order(index, weights, experts, every=False):
        seen.append(every)
        return real(index, weights, experts, every)

    monkeypatch.setattr(sops, "expert_order", order)
    moe = RoutedSquaredReluMoE(256, E, 2, 128, shared).to("cuda", torch.bfloat16)
    moe.router.data = moe.router.data.float()
    with torch.no_grad():
        moe(torch.randn(300, 256, device="cuda").bfloat16())
    assert seen == [together]
