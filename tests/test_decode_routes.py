"""Which decode steps are one launch from a product's sums on."""
import pytest
import torch

from kubeai_amd import ops


@pytest.mark.parametrize("rows,n_q,n_kv,hd,parts,dtype,takes", [
    (1, 32, 8, 128, 4, torch.bfloat16, True), (512, 32, 8, 128, 2, torch.bfloat16, True),
    (513, 32, 8, 128, 2, torch.bfloat16, False), (8, 8, 4, 256, 8, torch.bfloat16, True),
    (8, 32, 8, 128, 9, torch.bfloat16, False), (8, 32, 8, 128, 4, torch.float8_e5m2, False),
    (8, 28, 4, 128, 4, torch.bfloat16, False), (8, 8, 1, 256, 4, torch.bfloat16, False),
])
def test_sums_that_decode_attention_takes(rows, n_q, n_kv, hd, parts, dtype, takes):
    qkv = ops.ProductSums(torch.empty(parts, rows, (n_q + 2 * n_kv) * hd), None, None)
    cache = torch.empty(2, n_kv, 16, hd, dtype=dtype)
    cos_sin = torch.empty(16, hd)
    assert ops.decode_takes_sums(qkv, n_q, cos_sin, cache, cache) is takes
    assert not ops.decode_takes_sums(qkv.part[0], n_q, cos_sin, cache, cache)
