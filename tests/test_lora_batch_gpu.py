"""The batched LoRA kernels at the edges of their tiles: 16 tokens, 1024
inputs and 16 ranks a workgroup of the first, 256 outputs of the second.

y is rounded to bf16 once (2^-9 of itself); the sums before are fp32 over at
most 1100 + 64 terms (1100 * 2^-24 of the sum of magnitudes, far below)."""
import pytest
import torch

from kubeai_amd.engine.lora import LoRAManager, _float_word, _two_words

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _apply(T, H, out, ranks, ids, y_pad=0):
    from kubeai_amd import _C

    torch.manual_seed(T + H + out)
    x = torch.randn(T, H, device=DEV, dtype=torch.bfloat16)
    wide = torch.randn(T, out + y_pad, device=DEV, dtype=torch.bfloat16)
    y = wide[:, :out]
    sets = {lid: (torch.randn(r, H, device=DEV, dtype=torch.bfloat16) * 0.1,
                  torch.randn(out, r, device=DEV, dtype=torch.bfloat16), 2.0 / r)
            for lid, r in ranks.items()}
    table = torch.tensor([[A.data_ptr(), B.data_ptr(), _two_words(A.shape[0], lid), _float_word(s)]
                          for lid, (A, B, s) in sets.items()], dtype=torch.int64, device=DEV)
    want, rest = y.double(), wide[:, out:].clone()
    for t, lid in enumerate(ids):
        if lid in sets:
            A, B, s = sets[lid]
            want[t] += (B.double() @ (A.double() @ x[t].double())) * s
    _C.lora_apply(y, x, table, torch.tensor(ids, dtype=torch.int32, device=DEV),
                  max(ranks.values()))
    torch.testing.assert_close(y.double(), want, atol=1e-4, rtol=2.0 ** -8)
    assert torch.equal(wide[:, out:], rest)


@pytest.mark.parametrize("T", [1, 15, 16, 17, 50])
@pytest.mark.parametrize("H,out", [(1024, 512), (1032, 514), (40, 6), (2048, 511)])
def test_sizes(T, H, out):
    _apply(T, H, out, {3: 16, 9: 8}, [(0, 3, 9, 5)[t * 7 % 4] for t in range(T)])


@pytest.mark.parametrize("rank", [1, 7, 8, 17, 48, 64])
def test_ranks_beside_each_other(rank):
    _apply(33, 1024, 520, {1: rank, 2: 16, 3: 3}, [1, 2, 3] * 11)


def test_sixteen_adapters_in_a_tile_and_strided_rows():
    _apply(32, 256, 300, {k + 1: 8 + k % 9 for k in range(16)}, list(range(1, 17)) * 2, y_pad=5)
    _apply(20, 256, 300, {1: 16}, [0] * 20)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_an_adapter_without_finite_weights_keeps_to_its_tokens(bad):
    from kubeai_amd import _C

    torch.manual_seed(1)
    x = torch.randn(16, 64, device=DEV, dtype=torch.bfloat16)
    A = torch.randn(2, 8, 64, device=DEV, dtype=torch.bfloat16)
    B = torch.randn(2, 40, 8, device=DEV, dtype=torch.bfloat16)
    A[1, 3, 5] = B[1, 7, 2] = bad
    table = torch.tensor([[A[i].data_ptr(), B[i].data_ptr(), _two_words(8, i + 1),
                           _float_word(1.0)] for i in range(2)], dtype=torch.int64, device=DEV)
    ids = torch.tensor([1, 2] * 8, dtype=torch.int32, device=DEV)
    y = torch.zeros(16, 40, device=DEV, dtype=torch.bfloat16)
    _C.lora_apply(y, x, table, ids, 8)
    want = (x[::2].double() @ A[0].double().T) @ B[0].double().T
    torch.testing.assert_close(y[::2].double(), want, atol=1e-4, rtol=2.0 ** -8)
    assert not y[1::2].isfinite().any()


class _Cfg:
    hidden_size, intermediate_size, num_hidden_layers = 128, 256, 2
    num_attention_heads, num_key_value_heads, head_dim = 2, 1, 64
    num_local_experts = 0


class _Model(torch.nn.Module):
    cfg = _Cfg()


def test_manager_batched_equals_one_by_one():
    """The table's route against the per-adapter one, and what it leaves to it:
    ranks above the table's and tensors of another type."""
    m = LoRAManager(_Model(), DEV, torch.bfloat16)
    for lid in (4, 7):
        m.load(lid, None)
    ids = torch.tensor([4, 0, 7, 7, 4, 1], dtype=torch.int32, device=DEV)
    assert set(m._tables) == set(m.TARGETS)
    for target, din, dout in (("qkv", 128, 256), ("o", 128, 128), ("gate_up", 128, 512),
                              ("down", 256, 128)):
        x = torch.randn(6, din, device=DEV, dtype=torch.bfloat16)
        y = torch.randn(6, dout, device=DEV, dtype=torch.bfloat16)
        one, many = y.clone(), y.clone()
        m.apply(1, target, x, many, ids)
        tables, m._tables = m._tables, {}
        m.apply(1, target, x, one, ids)
        m._tables = tables
        torch.testing.assert_close(many, one, atol=1e-4, rtol=2.0 ** -7)
        assert torch.equal(many[1], y[1]) and torch.equal(many[5], y[5])
    m.unload(4)
    y2 = y.clone()
    m.apply(0, "down", x, y2, ids)
    assert torch.equal(y2[0], y[0]) and not torch.equal(y2[2], y[2])
    m.adapters[7]["qkv"][0] = (torch.zeros(65, 128, device=DEV, dtype=torch.bfloat16),
                               torch.zeros(256, 65, device=DEV, dtype=torch.bfloat16), 1.0)
    m._build_tables()
    assert "qkv" not in m._tables and "o" in m._tables


@pytest.mark.parametrize("pad,first", [(1, 0), (4, 0), (8, 3), (9, 1)])
@pytest.mark.parametrize("T", [1, 20])
def test_rows_that_begin_anywhere(T, pad, first):
    """x as a slice of wider rows, at any offset and stride."""
    m = LoRAManager(_Model(), DEV, torch.bfloat16)
    m.load(4, None)
    ids = torch.full((T,), 4, dtype=torch.int32, device=DEV)
    wide = torch.randn(T, 128 + pad, device=DEV, dtype=torch.bfloat16)
    x = wide[:, first : first + 128]
    y = torch.randn(T, 256, device=DEV, dtype=torch.bfloat16)
    A, B, s = m.adapters[4]["qkv"][1]
    want = y.double() + (x.double() @ A.double().T @ B.double().T) * s
    m.apply(1, "qkv", x, y, ids)
    torch.testing.assert_close(y.double(), want, atol=1e-4, rtol=2.0 ** -8)


def test_an_adapter_that_is_not_in_the_table_yet():
    """Put into the manager beside load() (as load() itself does before the table
    is rebuilt), and tensors that are let go: the table holds its own."""
    m = LoRAManager(_Model(), DEV, torch.bfloat16)
    m.load(4, None)
    kept = {t.data_ptr() for t in m._tables["qkv"][4]}
    assert kept == {t.data_ptr() for s in m.adapters[4]["qkv"] for t in s[:2]}
    m.adapters[9] = m._random_adapter(9)
    ids = torch.tensor([4, 9, 0], dtype=torch.int32, device=DEV)
    x = torch.randn(3, 128, device=DEV, dtype=torch.bfloat16)
    y = torch.zeros(3, 256, device=DEV, dtype=torch.bfloat16)
    m.apply(0, "qkv", x, y, ids)
    for t in (0, 1):
        A, B, s = m.adapters[int(ids[t])]["qkv"][0]
        want = (x[t].double() @ A.double().T @ B.double().T) * s
        torch.testing.assert_close(y[t].double(), want, atol=1e-4, rtol=2.0 ** -8)
    assert (y[2] == 0).all()


@pytest.mark.parametrize("rank", [1, 8, 33])
def test_infinite_weights_reach_the_output(rank):
    """An infinite B is infinite in y, with the sign of the product, also where
    the rank's value is one that bf16 holds exactly; NaN and 0 times it are NaN."""
    from kubeai_amd import _C

    x = torch.zeros(4, 64, device=DEV, dtype=torch.bfloat16)
    x[0, 0], x[1, 0], x[2, 0] = 1.0, -3.0, 0.0
    x[3] = torch.randn(64, device=DEV)
    A = torch.zeros(rank, 64, device=DEV, dtype=torch.bfloat16)
    A[0] = torch.randn(64, device=DEV)
    A[0, 0] = 0.5
    B = torch.randn(40, rank, device=DEV, dtype=torch.bfloat16)
    B[3, 0], B[5, 0], B[17, 0] = float("inf"), -float("inf"), float("nan")
    table = torch.tensor([[A.data_ptr(), B.data_ptr(), _two_words(rank, 1), _float_word(2.0)]],
                         dtype=torch.int64, device=DEV)
    y = torch.ones(4, 40, device=DEV, dtype=torch.bfloat16)
    want = y.double() + 2.0 * (x.double() @ A.double().T) @ B.double().T
    _C.lora_apply(y, x, table, torch.ones(4, dtype=torch.int32, device=DEV), rank)
    assert want[0, 3] == float("inf") and want[1, 3] == -float("inf") and want[2, 3].isnan()
    torch.testing.assert_close(y.double(), want, atol=1e-4, rtol=2.0 ** -8, equal_nan=True)


@pytest.mark.parametrize("T,out", [(1, 512), (17, 514), (50, 36), (97, 6144)])
def test_sums_take_the_adapters_in_their_first_part(T, out):
    """fp32 rows: nothing is rounded, so they are within the error of the fp32
    sums (1024 + 16 terms; 2^-14 of the magnitudes is above 1040 * 2^-24)."""
    from kubeai_amd import _C

    torch.manual_seed(T)
    ids = [(0, 3, 9, 5)[t * 7 % 4] for t in range(T)]
    x = torch.randn(T, 1024, device=DEV, dtype=torch.bfloat16)
    part = torch.randn(3, T, out, device=DEV)
    sets = {lid: (torch.randn(r, 1024, device=DEV, dtype=torch.bfloat16) * 0.1,
                  torch.randn(out, r, device=DEV, dtype=torch.bfloat16), 2.0 / r)
            for lid, r in ((3, 16), (9, 5))}
    table = torch.tensor([[A.data_ptr(), B.data_ptr(), _two_words(A.shape[0], lid), _float_word(s)]
                          for lid, (A, B, s) in sets.items()], dtype=torch.int64, device=DEV)
    want, size = part.double(), part.double().abs()
    for t, lid in enumerate(ids):
        if lid in sets:
            A, B, s = sets[lid]
            want[0, t] += (B.double() @ (A.double() @ x[t].double())) * s
            size[0, t] += (B.double().abs() @ (A.double().abs() @ x[t].double().abs())) * s
    _C.lora_apply(part[0], x, table, torch.tensor(ids, dtype=torch.int32, device=DEV), 16)
    assert ((part.double() - want).abs() <= size * 2.0 ** -14).all()
    assert torch.equal(part[1:].double(), want[1:])


def test_sums_of_a_product_with_adapters_equal_the_whole_one():
    """A projection as sums with the adapters in, against the product of bf16 rows
    with them added (rounded twice: 2^-8 of the larger of product and result)."""
    from kubeai_amd import ops
    from kubeai_amd.models.llama import EngineLinear, _project_adapted

    torch.manual_seed(0)
    m = LoRAManager(_Model(), DEV, torch.bfloat16)
    for lid in (4, 7):
        m.load(lid, None)
    fb = type("Batch", (), {})()
    fb.n_prefill = 1
    fb.lora_ids = torch.tensor([4, 0, 7, 7, 4, 1] * 20, dtype=torch.int32, device=DEV)
    lin = EngineLinear(256, 128, bias=False).to(DEV, torch.bfloat16).requires_grad_(False)
    x = torch.randn(120, 256, device=DEV, dtype=torch.bfloat16)
    for rows in (6, 24, 120):
        ids, fb.lora_ids = fb.lora_ids, fb.lora_ids[:rows].contiguous()
        whole = _project_adapted(lin, x[:rows], False, fb, m, 1, "down")
        as_sums = _project_adapted(lin, x[:rows], True, fb, m, 1, "down")
        fb.lora_ids = ids
        got = as_sums.part.sum(0) if isinstance(as_sums, ops.ProductSums) else as_sums
        assert rows > 96 or isinstance(as_sums, ops.ProductSums)
        size = 2.0 ** -8 * (whole.float().abs() + lin(x[:rows]).float().abs())
        assert ((got.float() - whole.float()).abs() <= size + 1e-4).all()


@pytest.mark.parametrize("T,inner", [(1, 8), (16, 248), (17, 264), (50, 1032)])
def test_gated_outputs(T, inner):
    """silu(gate) * up with the adapters in: one rounding to bf16 (2^-9 of the
    result); the kernel's exponential and quotient stay within 2^-20 of the value,
    the fp32 sums within 2^-14 of their magnitudes, which gate and up pass on with
    factors up to |up| * 1.1 and |silu(gate)|."""
    from kubeai_amd import _C

    torch.manual_seed(T)
    ids = [(0, 3, 9, 5)[t * 7 % 4] for t in range(T)]
    x = torch.randn(T, 264, device=DEV, dtype=torch.bfloat16)
    y = torch.randn(T, 2 * inner, device=DEV, dtype=torch.bfloat16)
    sets = {lid: (torch.randn(r, 264, device=DEV, dtype=torch.bfloat16) * 0.1,
                  torch.randn(2 * inner, r, device=DEV, dtype=torch.bfloat16), 2.0 / r)
            for lid, r in ((3, 16), (9, 5))}
    table = torch.tensor([[A.data_ptr(), B.data_ptr(), _two_words(A.shape[0], lid), _float_word(s)]
                          for lid, (A, B, s) in sets.items()], dtype=torch.int64, device=DEV)
    h, size, was = y.double(), y.double().abs(), y.clone()
    for t, lid in enumerate(ids):
        if lid in sets:
            A, B, s = sets[lid]
            h[t] += (B.double() @ (A.double() @ x[t].double())) * s
            size[t] += (B.double().abs() @ (A.double().abs() @ x[t].double().abs())) * s
    z = torch.empty(T, inner, device=DEV, dtype=torch.bfloat16)
    _C.lora_apply(y, x, table, torch.tensor(ids, dtype=torch.int32, device=DEV), 16, z)
    gate, up = h[:, :inner], h[:, inner:]
    silu = gate * torch.sigmoid(gate)
    want = silu * up
    bound = want.abs() * 2.0 ** -8 + 2.0 ** -14 * (
        1.1 * up.abs() * size[:, :inner] + silu.abs() * size[:, inner:]
    ) + 1e-6
    assert ((z.double() - want).abs() <= bound).all()
    assert torch.equal(y, was)


def test_gated_manager_equals_the_two_steps():
    """Against apply() and the activation, which round gate and up to bf16 first
    (2^-9 each, and 2^-9 of the result in both)."""
    from kubeai_amd import ops

    m = LoRAManager(_Model(), DEV, torch.bfloat16)
    m.load(4, None)
    ids = torch.tensor([4, 0, 1, 4, 4, 0], dtype=torch.int32, device=DEV)
    x = torch.randn(6, 128, device=DEV, dtype=torch.bfloat16)
    y = torch.randn(6, 512, device=DEV, dtype=torch.bfloat16)
    z = m.gated(1, x, y, ids)
    m.apply(1, "gate_up", x, y, ids)
    torch.testing.assert_close(z, ops.silu_and_mul(y), atol=1e-4, rtol=2.0 ** -6)
    assert m.gated(1, x, y[:, 1:], ids) is None
