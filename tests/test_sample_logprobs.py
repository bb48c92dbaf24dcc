"""Tokens and their log-probabilities out of one pass (ops.sample_with_logprobs)
against argmax / the noise's own reference and logsumexp in 64 bits."""
import pytest
import torch

from kubeai_amd import ops


def _logits(S, V, device, aligned=True):
    g = torch.Generator().manual_seed(S * 1000 + V)
    flat = torch.randn(S * V + 4, generator=g) * 5
    x = flat.to(device)[0 if aligned else 1 :][: S * V].view(S, V)
    if V > 4:
        x[0, 1:4] = float("-inf")  # masked tokens
    return x


def _check(x, tokens, logprobs):
    want = x.double() - torch.logsumexp(x.double(), -1, keepdim=True)
    want = want.gather(1, torch.tensor(tokens, device=x.device)[:, None])[:, 0].cpu()
    # sums of positive terms in fp32 (about 20 additions one after the other, then
    # trees) and a subtraction of numbers up to 64: 64 units of the last place
    got = torch.tensor(logprobs, dtype=torch.float64)
    assert torch.all((got - want).abs() <= 2.0**-24 * 64 * want.abs().clamp_min(1.0))


@pytest.mark.parametrize("S,V", [(1, 5), (3, 4097), (5, 256)])
def test_cpu(S, V):
    x = _logits(S, V, "cpu")
    tokens, logprobs = ops.sampled_to_host(ops.sample_with_logprobs(x))
    assert tokens == x.argmax(-1).tolist()
    _check(x, tokens, logprobs)


@pytest.mark.gpu
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("S,V", [(1, 1), (1, 5), (2, 131), (3, 4100), (40, 128256), (96, 131073)])
def test_gpu(S, V, aligned):
    x = _logits(S, V, "cuda", aligned)
    tokens, logprobs = ops.sampled_to_host(ops.sample_with_logprobs(x))
    assert tokens == x.argmax(-1).tolist()
    _check(x, tokens, logprobs)
    temps = torch.full((S,), 0.7, device="cuda")
    temps[::2] = 0.0
    seeds = torch.arange(S, device="cuda") + 9
    tokens, logprobs = ops.sampled_to_host(ops.sample_with_logprobs(x, temps, seeds, 3))
    assert tokens == ops.gumbel_sample(x, temps, seeds, 3).tolist()
    _check(x, tokens, logprobs)


@pytest.mark.gpu
def test_rows_of_one_value():
    x = torch.full((4, 1000), -3.0, device="cuda")
    x[1] = float("-inf")
    x[1, 999] = 1.0  # all other tokens masked: probability 1
    x[2] = float("nan")  # no token compares: none in the vocabulary is named
    x[3, 7] = float("inf")
    tokens, logprobs = ops.sampled_to_host(ops.sample_with_logprobs(x))
    assert tokens == [0, 999, 1000, 7] and logprobs[1] == 0.0
    assert abs(logprobs[0] + 6.907755279) < 1e-5
    assert all(v != v for v in logprobs[2:])


def test_fill_rows():
    out = torch.full((3, 4), 9, dtype=torch.int32)
    ops.fill_rows(out, [[1, 2], [], ])
    assert out.tolist() == [[1, 2, 0, 0], [0] * 4, [0] * 4]
    ops.fill_rows(out, [[1], [2, 3, 4, 5], [6]])
    assert out.tolist() == [[1, 0, 0, 0], [2, 3, 4, 5], [6, 0, 0, 0]]
    for rows in ([[1] * 5], [[1]] * 4):
        with pytest.raises((RuntimeError, IndexError)):
            ops.fill_rows(out, rows)


@pytest.mark.gpu
@pytest.mark.parametrize("S,V", [(1, 1), (3, 33), (70, 8192), (5, 65535), (5, 65536), (2, 65539)])
def test_tokens_alone(S, V):
    """One value at a time and 16 give the tokens of the pass with log-probabilities, the
    first of equal ones too."""
    x = _logits(S, V, "cuda")
    x[:, V // 2 :] = x[:, : V - V // 2]  # every value twice
    assert ops.greedy_sample(x).tolist() == x.argmax(-1).tolist()
    assert ops.greedy_sample(x).tolist() == ops.sampled_to_host(ops.sample_with_logprobs(x))[0]
    temps = torch.rand(S, device="cuda") + 0.2
    seeds = torch.arange(S, device="cuda")
    want = ops.sampled_to_host(ops.sample_with_logprobs(x, temps, seeds, 5))[0]
    assert ops.gumbel_sample(x, temps, seeds, 5).tolist() == want
