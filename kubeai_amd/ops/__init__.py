"""Op dispatch: hand-written gfx950 HIP kernels on GPU, torch reference on CPU.

Policy (deliberate, see repo instructions): on a ROCm GPU the HIP extension is
MANDATORY — if ``kubeai_amd._C`` failed to import, GPU-tensor calls raise
instead of silently falling back to eager PyTorch.  CPU tensors always use the
reference implementations (ref.py) so the engine logic is testable anywhere.
"""
from __future__ import annotations

import functools

import torch

from . import ref

_C = None
_C_IMPORT_ERROR: Exception | None = None
try:  # built in-tree by `python setup.py build_ext --inplace` / __graft_entry__.build()
    from kubeai_amd import _C  # type: ignore[attr-defined,no-redef]
except Exception as e:  # pragma: no cover - exercised only when ext missing
    _C_IMPORT_ERROR = e


def have_hip_ext() -> bool:
    return _C is not None


def _require_ext() -> None:
    if _C is None:
        raise RuntimeError(
            "kubeai_amd HIP extension (kubeai_amd._C) is not built but a GPU "
            "tensor reached the ops layer. Build it with "
            "`python setup.py build_ext --inplace` (PYTORCH_ROCM_ARCH=gfx950). "
            f"Original import error: {_C_IMPORT_ERROR!r}"
        )


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if isinstance(x, ProductSums):
        return _norm_sums(x, None, weight, eps, fp8=False)
    if x.is_cuda:
        _require_ext()
        out = torch.empty_like(x)
        _C.rmsnorm(out, x, weight, eps)
        return out
    return ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(x, residual, weight, eps: float):
    """In-place on GPU: x <- rmsnorm(x + residual), residual <- x + residual
    (x as ProductSums: a new tensor takes the norm)."""
    if isinstance(x, ProductSums):
        return _norm_sums(x, residual, weight, eps, fp8=False), residual
    if x.is_cuda:
        _require_ext()
        _C.fused_add_rmsnorm(x, residual, weight, eps)
        return x, residual
    return ref.fused_add_rmsnorm(x, residual, weight, eps)


def rope(q, k, positions, cos_sin):
    """In-place on GPU; returns (q, k)."""
    if q.is_cuda:
        _require_ext()
        _C.rope(q, k, positions, cos_sin)
        return q, k
    return ref.rope(q, k, positions, cos_sin)


def reshape_and_cache(k, v, k_cache, v_cache, slot_mapping) -> None:
    if k.is_cuda:
        _require_ext()
        if k_cache.dtype == torch.float8_e5m2:
            _C.reshape_and_cache_fp8(k, v, k_cache, v_cache, slot_mapping)
        else:
            _C.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)
        return
    ref.reshape_and_cache(k, v, k_cache, v_cache, slot_mapping)


def rope_takes_sums(k_cache, v_cache) -> bool:
    return (
        k_cache.is_cuda
        and k_cache.shape[3] % 16 == 0
        and k_cache.dtype in (torch.bfloat16, torch.float8_e5m2)
        and v_cache.dtype == k_cache.dtype
        and v_cache.shape == k_cache.shape
        and k_cache.is_contiguous()
        and v_cache.is_contiguous()
    )


def rope_and_cache(qkv, n_q: int, positions, cos_sin, k_cache, v_cache, slot_mapping):
    """q | k | v rows of the fused projection: q is rotated (in place on GPU) and
    returned as [T, n_q, hd], k is rotated and written to the paged cache with
    v. One launch on GPU where heads split into 16-byte units; qkv may be a
    product's sums there (rope_takes_sums)."""
    n_kv, hd = k_cache.shape[1], k_cache.shape[3]
    if isinstance(qkv, ProductSums):
        q = torch.empty((qkv.shape[0], n_q * hd), dtype=torch.bfloat16,
                        device=qkv.part.device)
        _C.rope_cache(q, positions, cos_sin, k_cache, v_cache, slot_mapping, n_q,
                      *qkv.args())
        return q.unflatten(-1, (n_q, hd))
    q, k, v = qkv.split([n_q * hd, n_kv * hd, n_kv * hd], dim=-1)
    q = q.unflatten(-1, (n_q, hd))
    if (
        qkv.is_cuda
        and hd % 16 == 0
        and qkv.dtype == torch.bfloat16
        and qkv.stride(1) == 1
        and qkv.stride(0) % 8 == 0
        and qkv.data_ptr() % 16 == 0
        and k_cache.dtype in (torch.bfloat16, torch.float8_e5m2)
        and v_cache.dtype == k_cache.dtype
        and v_cache.shape == k_cache.shape
    ):
        _require_ext()
        _C.rope_cache(qkv, positions, cos_sin, k_cache, v_cache, slot_mapping, n_q,
                      None, None, None)
        return q
    q, k = rope(q, k.unflatten(-1, (n_kv, hd)), positions, cos_sin)
    reshape_and_cache(k, v.unflatten(-1, (n_kv, hd)), k_cache, v_cache, slot_mapping)
    return q


def decode_plan(plans, seq_lens, block_tables, k_cache, window: int = 0, alone: bool = False):
    """How paged_attention_decode best splits rows of these lengths over caches like
    k_cache, worked out on the GPU once for all layers of a step: `plans` is the step's
    dict, which must not outlive it (None: no plan). A plan holds for the lengths that
    seq_lens had when it was made; recorded in a graph it is made again by each replay. How
    often a row is split follows from all rows' lengths, and so do the last bits of its
    result: beside other rows they may differ, as they do in steps of another size.

    Not for more than 512 rows, which take 135 us to plan (700; 40 rows 7, 200 17, 300 42,
    500 67), and where the rows are `alone` (no prompts in the step, whose launch with
    planned rows saves 5 us a layer and more) not for more than 256, nor where all see at
    most 128 keys and would not be split without a plan: the merge's launch is what a
    plan adds then (us, unplanned / planned: 76 rows of 11-22 4.3 / 5.8, 118 of 26-36 7.7 /
    10.1, 183 of 16-81 14.8 / 18.6; of 9 to 16 blocks as fast), or are few, where a plan's
    splits of eight tiles are too long (12 rows of 76-90 keys of one head of 256 8.4 / 9.5).
    Over 450 other batches of up to 400 rows planned ones take 0.78 of the time of the same
    number of splits each."""
    B, cols = seq_lens.shape[0], block_tables.shape[1]
    if plans is None or not seq_lens.is_cuda or not 1 <= B <= (256 if alone else 512):
        return None
    n_kv, bs, hd = k_cache.shape[1:]
    if window >= cols * bs:
        window = 0  # no row is longer
    if alone and min(cols * bs, window or cols * bs) <= 128:
        _require_ext()
        few = cols * bs <= 128 and B * n_kv <= 64
        if few or _C.paged_decode_splits(B, n_kv, hd, cols) == 1:
            return None
    key = (n_kv, hd, k_cache.element_size(), window)
    if key not in plans:
        _require_ext()
        plans[key] = _C.paged_decode_plan(seq_lens, *key)
    return plans[key]


def paged_attention_decode(
    q, k_cache, v_cache, block_tables, seq_lens, scale: float, out=None,
    window: int = 0, softcap: float = 0.0, plan=None,
):
    """q may be a row-strided view (fused qkv output); out must be
    contiguous (allocated here if not supplied). window > 0 enables
    sliding-window attention (Mistral/Gemma2 style: keys in
    (pos-window, pos]). plan: decode_plan of these lengths (another order of the
    sums)."""
    if q.is_cuda:
        _require_ext()
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.paged_attention_decode(
            out, q, k_cache, v_cache, block_tables, seq_lens, scale, window,
            softcap, None, plan
        )
        return out
    res = ref.paged_attention_decode(
        q, k_cache, v_cache, block_tables, seq_lens, scale, window=window,
        softcap=softcap,
    )
    if out is not None:
        out.copy_(res)
        return out
    return res


def decode_fp8_merges(n_q: int, splits: int) -> bool:
    """Whether the merge of a decode row's splits best converts the row to fp8 as
    well, where all rows have this many. One workgroup has the row then, and a wave of it
    merges a head for each 16 of the row, where the merge by itself has a wave per head
    (us with the attention, two launches / one: 16 heads 4 rows in 16 splits 16.0 / 14.3,
    72 rows in 2 13.2 / 10.9; 32 heads 38 rows of 400 in 2 splits 19.6 / 18.8, 7 rows of
    900 in 10 13.6 / 15.5, in 16 12.4 / 13.5; 64 heads 25 rows in 2 12.1 / 14.0, 2 in 12
    13.7 / 24.7). Planned splits, whose number the host does not know, are merged so up to
    32 heads: most rows have one or two (32 heads of 128, 38 rows of 400 22.5 / 21.3, 40 of
    100-700 23.2 / 22.1; long rows of few would rather be merged apart, one of 3000 11.6 /
    13.6)."""
    return splits > 1 and (n_q <= 16 or n_q <= 32 and splits <= 4)


def paged_attention_decode_fp8(
    q, k_cache, v_cache, block_tables, seq_lens, scale: float, window: int = 0,
    softcap: float = 0.0, plan=None,
):
    """quant_fp8 of paged_attention_decode's rows [B, n_q * hd]. On GPU the merge of
    a row's splits converts them, where that is the faster form."""
    B, n_q, hd = q.shape
    if not q.is_cuda or B == 0 or not (
        n_q <= 32 if plan is not None else decode_fp8_merges(
            n_q, _C.paged_decode_splits(B, k_cache.shape[1], hd, block_tables.shape[1])
        )
    ):
        out = paged_attention_decode(q, k_cache, v_cache, block_tables, seq_lens, scale,
                                     window=window, softcap=softcap, plan=plan)
        return quant_fp8(out.view(B, n_q * hd))
    out = torch.empty((B, n_q * hd), dtype=torch.float8_e4m3fn, device=q.device)
    out_scale = torch.empty(B, dtype=torch.float32, device=q.device)
    _C.paged_attention_decode(out, q, k_cache, v_cache, block_tables, seq_lens, scale,
                              window, softcap, out_scale, plan)
    return out, out_scale


def decode_takes_sums(qkv, n_q: int, cos_sin, k_cache, v_cache) -> bool:
    """Whether paged_attention_decode_sums takes these. Every split of a row adds the row's
    sums again, so not more than 512 rows, which fill the chip in a rotation of their own
    (us, that and the attention / one launch: 40/8 heads, 810 rows of 5-75 keys 50.9 / 60.6, 4/1
    heads 520 of 136-1436 53.9 / 57.7; over 250 steps of up to 512 rows 0.79, 1.03 at
    most)."""
    return (
        isinstance(qkv, ProductSums)
        and qkv.part.shape[1] <= 512
        and k_cache.dtype == v_cache.dtype == torch.bfloat16
        and k_cache.shape == v_cache.shape
        and k_cache.shape[2] == 16
        and k_cache.shape[3] in (128, 256)
        and n_q % k_cache.shape[1] == 0
        and n_q // k_cache.shape[1] in (1, 2, 4, 5, 6, 8)
        and (n_q // k_cache.shape[1] + 2) * k_cache.shape[3] <= 2048
        and qkv.part.shape[0] <= 8
        and cos_sin.dtype == torch.float32
        and cos_sin.is_contiguous()
        and aligned(cos_sin)
    )


def paged_attention_decode_sums(
    qkv, n_q: int, positions, cos_sin, slot_mapping, k_cache, v_cache, block_tables, seq_lens,
    scale: float, window: int = 0, softcap: float = 0.0, plan=None, fp8: bool = False,
):
    """rope_and_cache and paged_attention_decode in one launch (GPU only), for rows whose
    q | k | v is a product's sums: [B, n_q, hd] bf16, or (fp8) quant_fp8 of its rows. Every
    row's slot is the place of its last key (negative: nothing is written, and the cache
    has the key), and no other row reads that place."""
    B, (n_kv, _, hd) = qkv.shape[0], k_cache.shape[1:]
    merges = fp8 and (
        n_q <= 32 if plan is not None
        else decode_fp8_merges(n_q, _C.paged_decode_splits(B, n_kv, hd, block_tables.shape[1]))
    )
    dev = k_cache.device
    out = torch.empty((B, n_q, hd), device=dev,
                      dtype=torch.float8_e4m3fn if merges else torch.bfloat16)
    out_scale = torch.empty(B, dtype=torch.float32, device=dev) if merges else None
    _C.paged_attention_decode_sums(
        out, *qkv.args(), n_q, positions, cos_sin, slot_mapping, k_cache, v_cache,
        block_tables, seq_lens, scale, window, softcap, out_scale, plan)
    if not fp8:
        return out
    flat = out.view(B, n_q * hd)
    return (flat, out_scale) if merges else quant_fp8(flat)


def step_attention_takes(q, n_decode: int, k_cache, plan) -> bool:
    """Whether paged_attention_step has a step of these queries [T, n_q, hd]."""
    n_kv = k_cache.shape[1]
    return (
        plan is not None  # (on the GPU)
        and 0 < n_decode < q.shape[0]
        and q.shape[2] == 128
        and q.dtype == torch.bfloat16
        and q.stride(1) == 128 and q.stride(2) == 1
        and q.shape[1] in (n_kv, 2 * n_kv, 4 * n_kv, 8 * n_kv)
    )


def paged_attention_step(
    q, n_decode: int, k_cache, v_cache, decode_tables, decode_lens, prompt_tables,
    query_start_loc, prompt_lens, scale: float, window: int = 0, softcap: float = 0.0,
    plan=None, fp8: bool = False,
):
    """paged_attention_decode of the first n_decode rows and paged_attention_prefill of
    the others in one launch (step_attention_takes): [T, n_q, hd] bf16, or (fp8)
    quant_fp8 of its rows. Up to 1024 rows of up to 32 heads the merge of the decode rows'
    splits converts them; its workgroup a row is the slower conversion of many (us, with
    the attention, merge and conversion apart / one: 572 rows 41 / 38.8, 1501 rows 62 /
    62.3, 2008 rows 80 / 86, 6040 rows 371 / 393)."""
    T, n_q, hd = q.shape
    merges = fp8 and n_q <= 32 and T <= 1024
    out = torch.empty((T, n_q, hd), device=q.device,
                      dtype=torch.float8_e4m3fn if merges else torch.bfloat16)
    out_scale = torch.empty(T, dtype=torch.float32, device=q.device) if merges else None
    _C.paged_attention_step(
        out, out_scale, q, n_decode, k_cache, v_cache, decode_tables, decode_lens, plan,
        prompt_tables, query_start_loc, prompt_lens, scale, window, softcap)
    if not fp8:
        return out
    flat = out.view(T, n_q * hd)
    return (flat, out_scale) if merges else quant_fp8(flat)


def paged_attention_prefill(
    q, k_cache, v_cache, block_tables, query_start_loc, seq_lens, scale: float,
    out=None, window: int = 0, softcap: float = 0.0,
):
    if q.is_cuda:
        _require_ext()
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.paged_attention_prefill(
            out, q, k_cache, v_cache, block_tables, query_start_loc, seq_lens,
            scale, window, softcap
        )
        return out
    res = ref.paged_attention_prefill(
        q, k_cache, v_cache, block_tables, query_start_loc, seq_lens, scale,
        window=window, softcap=softcap,
    )
    if out is not None:
        out.copy_(res)
        return out
    return res


def silu_and_mul(x):
    if x.is_cuda:
        _require_ext()
        T, two_i = x.shape
        out = torch.empty((T, two_i // 2), dtype=x.dtype, device=x.device)
        _C.silu_and_mul(out, x)
        return out
    return ref.silu_and_mul(x)


def gelu_and_mul(x):
    """GeGLU (gemma family): gelu_tanh(gate) * up over packed [T, 2I]."""
    if x.is_cuda:
        _require_ext()
        T, two_i = x.shape
        out = torch.empty((T, two_i // 2), dtype=x.dtype, device=x.device)
        _C.gelu_and_mul(out, x)
        return out
    return ref.gelu_and_mul(x)


class ProductSums:
    """A matrix product of few rows whose parts along K are not added yet: fp32
    [parts, M, N], with the scales of fp8 operands. What reads it next adds,
    scales and rounds it to bf16 on the way (fused_add_rmsnorm, rmsnorm and
    their fp8 forms, rope_and_cache)."""

    is_cuda = True

    def __init__(self, part, x_scale=None, w_scale=None):
        self.part, self.x_scale, self.w_scale = part, x_scale, w_scale
        self.shape = part.shape[1:]

    def args(self):
        return self.part, self.x_scale, self.w_scale


_forward_ad = torch.autograd.forward_ad
_PLAIN_TENSORS = (torch.Tensor, torch.nn.Parameter)


def observed(*tensors) -> bool:
    """Whether something follows the tensors' operations that a kernel launch
    would pass by: autograd, forward mode, vmap, a trace or dispatch mode,
    autocast, a tensor subclass. Where the library's own operation stood by
    itself before, it still does then."""
    if (
        torch._C._len_torch_dispatch_stack()
        or _forward_ad._current_level >= 0
        or torch._C._functorch.peek_interpreter_stack() is not None
        or torch._C._get_tracing_state() is not None
        or torch.is_autocast_enabled("cuda")
    ):
        return True
    grad = torch.is_grad_enabled()
    for t in tensors:
        if type(t) not in _PLAIN_TENSORS or grad and t.requires_grad:
            return True
    return False


def aligned(*tensors) -> bool:
    """Whether kernels may read the tensors' storage 16 bytes at a time. (A slice
    that counts as contiguous can begin anywhere.)"""
    return all(t.data_ptr() % 16 == 0 for t in tensors)


def _skinny_operands(x, weight) -> bool:
    """Operands that the weight-streaming product takes."""
    return (
        _C is not None
        and x.is_cuda
        and x.dtype == weight.dtype
        and x.dtype in (torch.bfloat16, torch.float8_e4m3fn)
        and x.dim() == 2
        and 1 <= x.shape[0] <= 96
        and x.is_contiguous()
        and weight.is_contiguous()
        # (the stride of a single row may be anything)
        and x.stride(0) == x.shape[1]
        # (the library refuses fp8 columns that are no multiple of 16)
        and weight.shape[0] % (8 if x.dtype == torch.bfloat16 else 16) == 0
        and weight.shape[1] * weight.element_size() % 64 == 0
        and weight.shape[1] * weight.element_size() < 2**23
        and weight.device == x.device
        and not (torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad))
        and x.data_ptr() % 16 == weight.data_ptr() % 16 == 0
    )


def product_sums(x, weight, x_scale=None, w_scale=None):
    """x weight^T as ProductSums for a consumer that takes them, or None for
    operands that the kernel does not take (from 16384 columns on the product
    fills the chip without being cut). Whether it is the better form:
    sums_better."""
    if not (
        x.shape[0] <= 96 and weight.shape[0] < 16384 and _skinny_operands(x, weight)
    ):
        return None
    return ProductSums(_C.skinny_sums(x, weight), x_scale, w_scale)


def sums_better(
    M: int, N: int, K: int, fp8: bool, rope: bool = False, eager: bool = False
) -> bool:
    """Whether a product as ProductSums and the norm that adds them (rope: the
    rotation and cache write) beat the library's product and its reader. The
    reader's cost grows with parts x M x N, so wide products of many rows are the
    library's, and so are those that it cuts along K itself; eight-bit weights
    are read in half the time and leave less to gain. (In a whole decode step of 40
    rows in fp8 the sums of the products around attention gain 3 us a layer that
    pairs timed by themselves do not show.) us, weights out of cache,
    library / this: bf16 4096 -> 4096 8 rows 18.8 / 13.0, 96 rows 25.5 / 19.6;
    14336 -> 4096 8 rows 29.3 / 28.0, 40 rows 39.8 / 33.0; 4096 -> 6144 8 rows 17.5
    / 16.0 (rotation), 64 rows 21.0 / 21.9; 8192 -> 8192 33.5 / 39.4; 8192 -> 1024
    8 rows 14.8 / 10.7. fp8 4096 -> 4096 16 rows 16.1 / 11.0; 14336 -> 4096 40 rows
    24.9 / 21.4; 8192 -> 8192 8 rows 47.0 / 23.8, 16 rows 20.7 / 24.2.
    The line was drawn where this form and its reader were 1 to 4 us slower than they
    are, so it is a cautious one: of 22943 products at random (1 to 96 rows, 512 to
    12288 columns, K 512 to 28672, either reader) the 13496 that this rule and
    few_tiled_better choose take 0.52 of the library's time, 1.29 at worst (174 of them
    more than 1.05), and of the other 9447 two thirds would be 5 % or more faster as
    sums, 0.83 of the time in all: fp8 4096 -> 4096 64 rows 16.6 / 15.4, 512 -> 4096 8 rows
    8.6 / 7.2. (bf16 8192 -> 1024 of 40 rows, not this rule's either, few_tiled_better
    has: 15.3, streaming 12.4, tiled 14.3.)
    eager: the step is not replayed from a graph, so the host's launches bound it
    while the weights are small, and the library's call takes 10 us of the host
    more (80 tokens of a prompt on 8 layers of 4096: 1796 us / 1493)."""
    if eager and N * K * (1 if fp8 else 2) < 2**26:
        return True
    if K > 16384 and N <= 6144:  # (there the library is two to four times slower)
        return True
    if fp8:
        if rope and (K < 2048 or M > 48 or M > 16 and 2048 < K < 4096):
            return False
        if K < 2048:
            return M <= 40 and N <= 2304 if K >= 1024 and M > 32 else (
                M <= 32 and N <= (2304 if K < 1024 else 5120)
            )
        if M <= 12:
            return N <= 4096 or K <= 4096 or N >= 8192
        if N > 4096:
            return N <= 6144 and K <= 4096 if rope else (
                M <= 32 and K <= 2048 and N <= 8192
            )
        if M <= 48:
            return True
        return (N <= 3072 or K > 4096) if M <= 64 else K >= 12288
    if K <= 1024:
        return (N <= 6144 or M <= 48) and not (rope and K < 1024 and 1024 < N <= 4096)
    if N > 6144:
        return False
    if K <= 4096:
        if N > 4096:
            if rope and (M <= 16 or 32 < M <= 48):
                return True
            return M <= (48 if K <= 2048 else 8)
        return M <= 64 or min(N, K) >= 3072
    if M <= 16:
        return N <= 2048 or K >= 12288 and N <= 4096
    return N <= 4096 if M <= 32 else N >= 2048


def _even_rows(K: int, fp8: bool) -> bool:
    """Whether weight rows lie whole 4 KB apart: the same columns of all of them are
    then the same few channels of the memory. Kernels that begin at columns apart
    (csrc/skinny_gemm.hip, csrc/tiled_gemm.h) lose less to that than the library's."""
    return K * (1 if fp8 else 2) % 4096 == 0


def _streams_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether the weight-streaming product beats the library's. us, weights out of
    cache, library / this. Up to 16 rows and a width that fills the chip, uncut (8 rows):
    bf16 4096 -> 28672 60.2 / 41.0, 4096 -> 16384 32.1 / 23.5, 8192 -> 24576 82 / 71, 4096 ->
    128256 187 / 173, 8192 -> 57344 172 / 158, 2304 -> 87808 136 / 80; but 1792 -> 56320 38.6
    / 39.8, 2304 -> 256000 207 / 218; fp8 4096 -> 28672 31.7 / 23.6, 4096 -> 16384 26.4 /
    14.0, 4096 -> 128256 112 / 94, but 9472 -> 59648 102 / 110, 1536 -> 116992 39 / 41.
    Beyond 40000 columns only where rows lie whole 4 KB apart, or the CUs have even
    shares of the columns' tiles (bf16 2304 -> 49152 48.9 / 43.7, but 49536 at 13 rows 43.3 /
    50.8; fp8 1920 -> 49152 20.6 / 20.0, 53504 21.7 / 23.1), or they are so many that the last
    share counts little. Over 308 products the 200 chosen took 0.74 of the time, 1.10 at
    worst; of 130 others beside 49152 and 65536 columns 0.87, 1.13 at worst.
    fp8 from 8192 columns on up to 12 rows, cut along K (6656 -> 9216 38 / 19, 8192 -> 8192
    16 rows 16.4 / 21.3); bf16 of such widths not (7680 -> 14848 45 / 52). Rows
    under 256 bytes stay: one launch against another (128 -> 65536 fp8 5.4 / 5.1).
    Very long rows, which the library does not cut: 32256 -> 2048 83 / 32 at 8 rows, 127 /
    52 at 96. It does at 16384, where the line lies by a kernel that took a third longer
    (-> 1024 bf16 16 rows 21.0 / 16.4, fp8 64 rows 26.4 / 14.5; left to the library: bf16 48
    rows 21.3 / 19.2, -> 2048 fp8 96 rows 21.6 / 17.5)."""
    if K >= 8 * N and K >= 16384:
        return K > 16384 or M <= (64 if fp8 else 32)
    if M > 16 or K * (1 if fp8 else 2) < 256:
        return False
    if N < 16384:
        return fp8 and N >= 8192 and M <= 12
    if N <= 40000 or _even_rows(K, fp8):
        return True
    even_shares = N % 16384 == 0 and N <= 65536
    if fp8:
        return K <= 1024 or even_shares and K <= 8192
    return 65536 <= N < 200000 or even_shares and K <= (6144 if M <= 8 else 4096)


def _tiled_operands(x, weight) -> bool:
    """Operands that the tiled product takes (and the library, which refuses fp8
    columns that are no multiple of 16)."""
    es = x.element_size()
    return (
        _C is not None
        and x.is_cuda
        and weight.device == x.device
        and x.dtype == weight.dtype
        and x.dtype in (torch.bfloat16, torch.float8_e4m3fn)
        and x.dim() == weight.dim() == 2
        and x.shape[0] >= 1
        and x.shape[1] == weight.shape[1]
        and x.is_contiguous()
        and weight.is_contiguous()
        and weight.shape[1] * es % 128 == 0
        and weight.shape[1] * es < 2**23
        and weight.shape[0] % 16 == 0
        and not observed(x, weight)
        and aligned(x, weight)
    )


def _row_and_column_scales(x, weight, x_scale, w_scale) -> bool:
    """Scales of fp8 operands that the kernels read: one per row and column, dense
    fp32. (The library takes one for all as well.)"""
    return (
        x_scale.dtype == w_scale.dtype == torch.float32
        and x_scale.device == w_scale.device == x.device
        and x_scale.numel() == x.shape[0]
        and x_scale.is_contiguous()
        and w_scale.numel() == weight.shape[0]
        and w_scale.is_contiguous()
        and not observed(x_scale, w_scale)
    )


def _tiled_scales(x, weight, x_scale, w_scale) -> bool:
    """Scales that the tiled product reads, the columns' four at a time."""
    return (
        _row_and_column_scales(x, weight, x_scale, w_scale)
        and w_scale.shape == (1, weight.shape[0])
        and aligned(w_scale)
    )


def _kernel_writes(out, x, weight) -> bool:
    """Whether a kernel writes the product into `out` (None: a new tensor). (The
    library fits one of another shape to the result.)"""
    return out is None or (
        out.shape == (x.shape[0], weight.shape[0]) and out.is_contiguous()
        and out.dtype == torch.bfloat16 and out.device == x.device
    )


def _kernel_adds(bias, weight) -> bool:
    return bias is None or (
        bias.dtype == torch.bfloat16 and bias.device == weight.device
        and bias.numel() == weight.shape[0] and bias.is_contiguous()
        and not observed(bias)
    )


def _tiled_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether the tiled product (csrc/tiled_gemm.h) beats the library's. fp8: from
    97 rows on, unless K is short, where the stores count (us, weights out of
    cache, library / this: 16384 x 512 8192 rows 104 / 127, 1024 x 1024 4.8 / 5.8), or
    the smallest tiles (64 x 128) are fewer than 160 and leave CUs idle, where the
    library cuts K (256 x 11776 775 rows 15.9 / 32.7, 6144 x 4096 97 rows 15.9 / 17.1,
    4096 x 14336 256 rows 34 / 49; 7168 x 5632 148 rows, 168 tiles, 22.3 / 21.4), which
    it does up to K 16384 (1504 x 18304 353 rows, 72 tiles, 77 / 56); or its tile of 256
    rows is almost full beside many columns (28672 x 4096 256 rows 40.4 / 40.7, 260
    rows 56 / 43). Over 400 others (97 to 6000 rows, 256 to 32768 columns, K 2048 to
    20000) the chosen ones take 0.77 of the library's time, 1.05 at worst. Logits: 128256 x
    4096 fp8 40 rows 129 / 107, 96 rows 121 / 118, bf16 40 rows 203 / 192, 160
    rows 246 / 213, 384 rows 437 / 339, 1024 rows 853 / 838; 57344 x 8192 fp8 40 rows
    126 / 90; over 68 others 0.85, in bf16 above 200 rows 0.82 to 1.10. 17 to
    96 rows beside 24576 columns and more of even rows (fp8 28672 x 4096 40 rows 31.6 / 25.7,
    96 rows 33.1 / 28.9; bf16 57.1 / 45.4 and 58.8 / 49.6, but 57344 x 8192 173 / 163, 16384
    x 4096 34.8 / 40.5). fp8 rows of other lengths where the library's tiles do not fill:
    18432 to 32767 columns however short they are (22016 x 1280 36 rows 11.7 / 10.2, 18432 x
    128 40 rows 5.2 / 4.8, 32000 x 256 8.5 / 5.7; over 117 products 0.83, 1.06 at worst) and
    from 45056 on (58368 x 2560 43.6 / 34.4; over 25 with K from 1024 0.75, 1.14 at
    worst), but 35840 x 2048 21.1 / 23.8. bf16 beside 65536 columns (96256 x 2304 36 rows
    95 / 86, 91392 x 3264 132 / 124; over 41 products 0.79, 1.02 at worst), but 49920 to 65152
    columns 0.89 to 1.10. Other bf16 products stay (28672 x 4096 2048 rows 333 / 391)."""
    if M <= 16:
        return False
    if M <= 96:
        even = N >= 24576 and _even_rows(K, fp8)
        if fp8:
            return even or 18432 <= N < 32768 or N >= 45056 and K >= 1024
        if N >= 98304 and K >= 2048:
            return True
        return K <= 4096 and (even or 65536 <= N < 200000)
    if N >= 49152 and K >= 2048:
        return fp8 or M <= 1024 and N >= 98304
    tiles = -(-M // 64) * -(-N // 128)
    if K > 16384:
        return fp8 and tiles >= 64
    return fp8 and K >= 2048 and tiles >= 160 and not (192 < M <= 256 and N >= 16384)


def fp8_product_tiled(M: int, N: int, K: int) -> bool:
    """Whether linear_fp8 has a product of these sizes, without a bias, from the tiled
    kernel and not from the library."""
    return N % 16 == 0 and K % 128 == 0 and K < 2**23 and _tiled_better(M, N, K, fp8=True)


def _tiled_linear(x, weight, x_scale=None, w_scale=None, out=None, act=0):
    if out is None:
        out = torch.empty(
            (x.shape[0], weight.shape[0] // (2 if act else 1)), dtype=torch.bfloat16,
            device=x.device,
        )
    _C.tiled_linear(out, x, weight, x_scale, w_scale, act)
    return out


def gated_better(M: int, N: int, K: int) -> bool:
    """Whether tiled_gated beats the library's bf16 product and the activation: up to
    512 rows, with short K up to 1024 (us, those / tiled_gated: 28672 x 4096 128 rows
    58.4 / 56.2, 384 rows 88 / 83, 640 rows 150 / 160, 2048 rows 381 / 408; 18432 x 2304
    gelu 384 rows 45.9 / 41.4, 1024 rows 102 / 94, 2048 rows 172 / 181, 5376 rows 399 /
    382 alone but 379 / 385 in a model). Not two row tiles of few columns, which leave
    CUs idle (9216 x 7680 126 rows 53 / 60), and not rows that almost fill the library's
    tile of 256 (17280 x 6656 195 rows 82 / 91, 28672 x 4096 256 rows 70 / 69). Over 79
    others (97 to 1024 rows, 8192 to 40000 columns, K 2048 to 8192) 0.89 of the time,
    1.06 at worst."""
    return 96 < M and N >= 8192 and K >= 2048 and (M <= 512 or K <= 2560 and M <= 1024) and (
        M > 128 or N > 10240
    ) and not (192 < M <= 256 and K > 2560)


def tiled_gated(x, weight, gelu=False):
    """silu_and_mul (gelu: gelu_and_mul) of x weight^T in bf16 (weight: gate rows,
    then up rows) in one launch, the activation in fp32 and rounded once; None where
    the product is not a tiled one or two launches are faster."""
    (M, K), N = x.shape, weight.shape[0]
    if not (
        gated_better(M, N, K)
        and x.dtype == torch.bfloat16
        and weight.dim() == 2 and N * weight.stride(0) * 2 < 2**31
        and _tiled_operands(x, weight)
    ):
        return None
    return _tiled_linear(x, weight, act=2 if gelu else 1)


def gated(x, weight, gelu=False):
    """What tiled_gated computes, also up to 96 rows: by the weight-streaming kernel or
    the tiled one where linear has the product, uncut, from them (28672 x 4096 one row:
    product 41.2 us, this 42.0, the activation's launch 4.7); None where two launches
    are faster."""
    (M, K), N = x.shape, weight.shape[0]
    if M > 96:
        return tiled_gated(x, weight, gelu)
    if x.dtype != torch.bfloat16 or weight.dim() != 2 or N * K * 2 >= 2**31:
        return None
    if (
        M <= 16 and N >= 16384  # (uncut)
        and _streams_better(M, N, K, fp8=False)
        and not observed(x, weight)
        and _skinny_operands(x, weight)
    ):
        y = torch.empty((M, N // 2), dtype=x.dtype, device=x.device)
        _C.skinny_gated(y, x, weight, 2 if gelu else 1)
        return y
    if _tiled_better(M, N, K, fp8=False) and _tiled_operands(x, weight):
        return _tiled_linear(x, weight, act=2 if gelu else 1)
    return None


#: Products of more rows are not handed on as sums: whole ones fill the chip.
MAX_SUM_ROWS = 2048


@functools.lru_cache(maxsize=4096)
def tiled_sums_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether a product of more than 96 rows as ProductSums of a tiled product
    that is cut along K, and the norm or rotation that adds them, beat the product
    as a whole and its reader: where its tiles alone leave CUs idle. By the costs
    of both (csrc/tiled_gemm.hip) and 3.5 us that a reader of few rows takes longer.
    (In bf16 the library's product is the other form; the tiled one's cost stands for
    it.) Over 160 products (97 to 2048 rows, 512 to 12288 columns, K 1024 to 28672) with
    the norm, the chosen ones take 0.60 (fp8) and 0.62 (bf16) of the time, 1.0 at worst;
    over 190 others with either reader 1.1 at worst (us with the
    norm: 4096 x 14336 128 rows fp8 51 / 26, bf16 76 / 35; 512 rows 53 / 49, 92 / 70; 1024
    rows bf16 139 / 116; 4096 x 4096 128 rows bf16 28 / 19, fp8 15.5 / 16.7: whole)."""
    es = 1 if fp8 else 2
    if _C is None or not 96 < M <= MAX_SUM_ROWS or not 0 < N <= 16384 or (
        K < 1 or K * es % 128
    ):
        return False
    whole = _C.tiled_plan(M, N, K * es, fp8, False)[2]
    return _C.tiled_plan(M, N, K * es, fp8, True)[2] + 3.5 < 0.95 * whole


def few_tiled_better(M: int, N: int, K: int, fp8: bool, rope: bool, sums: bool) -> bool:
    """Whether a product of 17 to 96 rows is best read as the sums of the tiled
    product. sums: the streaming product's sums beat the library's (sums_better);
    there the streaming kernel is the slower one where K is long or the rows are
    many (us with the norm, streaming / tiled: fp8 4096 x 14336 24 rows 23.3 / 20.7,
    96 rows 28.9 / 24.0; 4096 x 4096 24 rows 13.8 / 14.2, 40 rows 15.4 / 13.4; 2048 x
    2048 24 rows 8.8 / 9.8, 96 rows 12.0 / 11.2; bf16 4096 x 14336 96 rows 39.9 / 31.8).
    Up to 32 rows of up to 2048 columns a tile is half empty and few of them are
    there (896 x 11008 22 rows 12.6 / 13.3, 1664 x 5888 21 rows 12.4 / 13.4; K 17920 15.8 / 15.3).
    Else the library's product and reader / this: fp8 3072 x 8192 40 rows 17.1 / 16.0
    (rotation 16.9 / 17.0), 96 rows 25.4 / 17.8; 8192 x 28672 40 rows 74 / 52; 8192 x
    8192 40 rows 22.6 / 24.7; bf16 6144 x 4096 40 rows 20.4 / 17.9, 96 rows 25.9 / 20.7;
    10240 x 8192 24 rows 41.1 / 40.7, 96 rows 54.9 / 42.9; 2304 x 2048 80 rows 12.0 /
    12.6. Over 200 products (512 to 12288 columns, K 1024 to 28672) with the norm, the
    chosen ones take 0.83 (fp8) and 0.73 (bf16) of the other form's time, 1.01 at
    worst; over 160 beside the edges 0.83, 1.07 at worst. Beyond the edges lie widths
    of served models at which the library's product is the better one (it has tuned
    ones for them); at most widths between it is not (0.55 to 1.0 over 180 products)."""
    if sums:
        if M <= 32 and N <= 2048 and K <= 16384:
            return False
        return K >= 8192 or K >= 4096 and (M >= 32 or N > 4096) or K >= 2048 and M >= 80
    if K >= 16384:
        return True
    if fp8:
        return K >= 8192 and (
            N <= 2304 and M <= 64 or N <= 4096 and (M >= 24 and not rope or K >= 12288)
            or N > 8192 and M >= 40
        )
    return K >= 4096 and N <= 6144 or K >= 8192 and M >= 40 and N > 8192 or (
        K >= 2304 and M >= 80 and 2304 < N <= 4096
    )


@functools.lru_cache(maxsize=4096)
def narrow_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether a product of up to 64 rows is best read as the sums of tiles of 64 columns
    (csrc/tiled_gemm.hip: narrow_sums): their workgroups, one a CU at most, leave few CUs
    idle, and K is more than a few steps for each. Measured against the form that the rules
    below have without this one, weights out of cache (us, that form / narrow tiles: fp8
    6144 x 4096 40 rows with the norm 17.8 / 14.3, bf16 2304 x 9216 1 row 20.5 / 14.6). Left:
    - bf16 with 192 workgroups (6144 x 4096 40 rows 18.4 / 19.8), fewer of them (8256 x 9344
      44 rows 39 / 54), few steps (fp8 2048 x 2048 8 rows 7.3 / 8.3).
    - eight parts, which are no fewer than the streaming product's, up to 32 rows (over 175
      products with either reader 1.04, 1.13 at worst; bf16 2048 x 4096 3 rows 9.3 / 10.3).
    - one part, of more than 8192 columns, where the library has tuned products (bf16 14336 x
      8192 1 row 51.5 / 57.3, 16384 x 8192 64 rows 61 / 71), the streaming one is uncut (fp8
      16384 x 4096 8 rows 21.6 / 23.7) or wider tiles are taken (fp8 12672 x 20480 55 rows
      1.22, bf16 13312 x 9216 62 rows 1.17).
    - long K beside more than 48 rows (fp8 7168 x 22528 51 rows 41.1 / 44.2), up to 16 rows
      bf16 in two parts with tuned library products (6784 x 12288 1 row 37.9 / 41.8) and fp8
      rows that all begin in one channel (4096 x 16384 1 row 19.4 / 21.7 with the rotation).
    Over 1400 products (1 to 64 rows, 512 to 16384 columns, K 640 to 24500) the chosen ones
    take, with the norm, 0.91 of the time of other sums and 0.80 of the library's product,
    with the rotation 0.93 and 0.81; 6 of 2329 take more than 1.07 (bf16 with the rotation
    4096 x 8192 2 rows 1.15, 3712 x 22016 5 rows 1.11). Read by decode attention (which
    reads them once for each of a row's splits) 0.91 over 90 products, 1.06 at worst (fp8 6144
    x 4096 1 row 18.1 / 19.0)."""
    if not 1 <= M <= 64 or N < 1:
        return False
    tiles, steps = -(-N // 64), K * (1 if fp8 else 2) // 128
    parts = min(8, 256 // tiles) if tiles <= 256 else 0
    if not (
        parts > 0
        and parts * tiles >= (192 if fp8 else 200)
        and steps >= parts * (5 if M > 16 else 7)
    ):
        return False
    if parts == 8:
        return M > 32
    if parts == 1:
        return K % 4096 != 0 and (M <= 16 or fp8 and K < 8192)
    if M <= 16:
        return K % 16384 != 0 if fp8 else parts > 2 or K % 4096 != 0
    return M <= 48 or K < 15000


def tiled_sums(x, weight, x_scale=None, w_scale=None):
    """x weight^T as ProductSums of the tiled product, cut along K so that it
    fills the chip (narrow_better: in tiles of 64 columns), or None for operands that it
    does not take."""
    if not _tiled_operands(x, weight) or x_scale is not None and observed(x_scale, w_scale):
        return None
    narrow = narrow_better(x.shape[0], *weight.shape, x.element_size() == 1)
    sums = _C.narrow_sums if narrow else _C.tiled_sums
    return ProductSums(sums(x, weight), x_scale, w_scale)


def sums_for_reader(x, weight, x_scale=None, w_scale=None, rope=False, eager=False):
    """x weight^T (fp8 with the scales of both) as ProductSums where that and the
    norm, or (rope) the rotation, that reads it are the fastest form, or None: the
    product as a whole. eager: see sums_better."""
    M, (N, K), fp8 = x.shape[0], weight.shape, x_scale is not None
    if M > 96:  # (in a trace sizes are tensors, which no rule is to keep)
        better = type(M) is int and tiled_sums_better(M, N, K, fp8)
        return tiled_sums(x, weight, x_scale, w_scale) if better else None
    if type(M) is int and narrow_better(M, N, K, fp8):
        got = tiled_sums(x, weight, x_scale, w_scale)
        if got is not None:
            return got
    sums = sums_better(M, N, K, fp8=fp8, rope=rope, eager=eager)
    if M > 16 and N < 16384 and few_tiled_better(M, N, K, fp8, rope, sums):
        got = tiled_sums(x, weight, x_scale, w_scale)
        if got is not None:
            return got
    return product_sums(x, weight, x_scale, w_scale) if sums else None


def linear(x, weight):
    """x weight^T. Few rows against a wide or a very long weight go through the
    weight-streaming kernel (csrc/skinny_gemm.hip), logits through the tiled one
    (csrc/tiled_gemm.h), the rest to the library."""
    if (
        x.dim() == weight.dim() == 2
        and x.shape[0] <= 96
        and x.is_cuda
        and _streams_better(x.shape[0], *weight.shape, fp8=False)
        and x.dtype == torch.bfloat16
        and not observed(x, weight)
        and _skinny_operands(x, weight)
    ):
        y = torch.empty(
            (x.shape[0], weight.shape[0]), dtype=x.dtype, device=x.device
        )
        _C.skinny_linear(y, x, weight, None, None, None)
        return y
    if (
        x.is_cuda
        and x.dim() == weight.dim() == 2
        and x.dtype == torch.bfloat16
        and _tiled_better(x.shape[0], *weight.shape, fp8=False)
        and _tiled_operands(x, weight)
    ):
        return _tiled_linear(x, weight)
    return torch.nn.functional.linear(x, weight)


def linear_fp8(xq, x_scale, weight, w_scale, bias=None, out=None):
    """(xq * x_scale) (weight * w_scale)^T + bias in bf16; xq [M, K] and weight
    [N, K] e4m3, x_scale [M], w_scale [1, N]; into `out` (dense rows) if given."""
    if (
        xq.shape[0] <= 96
        and _streams_better(xq.shape[0], *weight.shape, fp8=True)
        and not observed(xq, weight)
        and _skinny_operands(xq, weight)
        and _row_and_column_scales(xq, weight, x_scale, w_scale)
        and _kernel_adds(bias, weight)
        and _kernel_writes(out, xq, weight)
    ):
        if out is None:
            out = torch.empty(
                (xq.shape[0], weight.shape[0]), dtype=torch.bfloat16, device=xq.device
            )
        _C.skinny_linear(out, xq, weight, x_scale.view(-1), w_scale.view(-1), bias)
        return out
    if (
        bias is None
        and _tiled_better(xq.shape[0], *weight.shape, fp8=True)
        and _tiled_operands(xq, weight)
        and _tiled_scales(xq, weight, x_scale, w_scale)
        and _kernel_writes(out, xq, weight)
    ):
        return _tiled_linear(xq, weight, x_scale.view(-1), w_scale.view(-1), out)
    kw = {} if out is None else {"out": out}
    return torch._scaled_mm(
        xq, weight.t(), scale_a=x_scale.view(-1, 1), scale_b=w_scale, bias=bias,
        out_dtype=torch.bfloat16, **kw,
    )


def rmsnorm_fp8(x, weight, eps: float):
    """GPU-only: rmsnorm with fused per-row fp8 quantization."""
    _require_ext()
    if isinstance(x, ProductSums):
        return _norm_sums(x, None, weight, eps, fp8=True)
    out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
    _C.rmsnorm_fp8(out, scale, x, weight, eps)
    return out, scale


def fused_add_rmsnorm_fp8(x, residual, weight, eps: float):
    """GPU-only, in-place residual update; returns (fp8 out, row scales)."""
    _require_ext()
    if isinstance(x, ProductSums):
        return _norm_sums(x, residual, weight, eps, fp8=True)
    out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
    _C.fused_add_rmsnorm_fp8(out, scale, x, residual, weight, eps)
    return out, scale


def _norm_sums(x: ProductSums, residual, weight, eps: float, fp8: bool):
    """bf16 rows, or (fp8 rows, scales), of the norm of a product's sums."""
    dev = x.part.device
    out = torch.empty(
        x.shape, dtype=torch.float8_e4m3fn if fp8 else torch.bfloat16, device=dev
    )
    scale = torch.empty(x.shape[0], dtype=torch.float32, device=dev) if fp8 else None
    _C.rmsnorm_sums(out, scale, *x.args(), residual, weight, eps)
    return (out, scale) if fp8 else out


class BranchNorm:
    """A branch whose norm is still to be taken, by norm_add_norm of what reads it
    next (add_and_norm)."""

    def __init__(self, x, weight, eps: float):
        self.x, self.weight, self.eps = x, weight, eps
        self.shape = x.shape


def _norm_add_norm_takes(x, residual, w1, w2) -> bool:
    tensors = [residual, w2] + [t for t in (w1, x) if isinstance(t, torch.Tensor)]
    return (
        residual.is_cuda
        and residual.dim() == 2
        and x.shape == residual.shape
        and residual.shape[1] % 8 == 0
        and residual.shape[1] <= 16384
        and all(t.dtype == torch.bfloat16 and t.is_contiguous() for t in tensors)
        and all(w is None or w.shape == residual.shape[1:] for w in (w1, w2))
        and aligned(*tensors)
        and not observed(*tensors)
    )


def add_and_norm(x, residual, weight, eps: float):
    """hidden = x + residual in bf16 and its norm; returns (norm, hidden). x may be a
    BranchNorm (of a tensor or ProductSums), whose norm is added then. On GPU one
    launch, with the bits of rmsnorm, the addition and rmsnorm after one another."""
    w1 = None
    if isinstance(x, BranchNorm):
        if x.eps == eps and _norm_add_norm_takes(x.x, residual, x.weight, weight):
            x, w1 = x.x, x.weight
        else:
            x = rmsnorm(x.x, x.weight, x.eps)
    if not (w1 is not None or _norm_add_norm_takes(x, residual, None, weight)):
        hidden = x + residual
        return rmsnorm(hidden, weight, eps), hidden
    _require_ext()
    hidden, out = torch.empty_like(residual), torch.empty_like(residual)
    sums = x.args() if isinstance(x, ProductSums) else (None, None, None)
    _C.norm_add_norm(out, hidden, None if sums[0] is not None else x, *sums, residual,
                     w1, weight, eps)
    return out, hidden


def silu_and_mul_fp8(x):
    if not x.is_cuda:
        return ref.quant_fp8(ref.silu_and_mul(x))
    _require_ext()
    T, two_i = x.shape
    out = torch.empty((T, two_i // 2), dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty(T, dtype=torch.float32, device=x.device)
    _C.silu_and_mul_fp8(out, scale, x)
    return out, scale


def quant_fp8(x):
    if not x.is_cuda:
        return ref.quant_fp8(x)
    _require_ext()
    out = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty(x.shape[0], dtype=torch.float32, device=x.device)
    _C.quant_fp8(out, scale, x)
    return out, scale


def moe_route(x, router, top_k: int):
    """GPU-only: fp32 router scores of x [T, H] (router [E, H], both bf16) and
    the softmax over every token's top_k experts. Returns (weight fp32 [T, k],
    begin int32 [E + 1], src, place int32 [T k]): rows begin[e]..begin[e + 1] of
    the expert order are token src[row]'s, pair (t, j) is row place[t k + j]."""
    _require_ext()
    T, E, n = x.shape[0], router.shape[0], x.shape[0] * top_k
    i32 = torch.empty(3 * n + E + 1, dtype=torch.int32, device=x.device)
    index, src, place, begin = i32.split([n, n, n, E + 1])
    weight = torch.empty((T, top_k), dtype=torch.float32, device=x.device)
    _C.moe_route(index.view(T, top_k), weight, begin, src, place, x, router.detach())
    return weight, begin, src, place


def moe_combine(y, place, weight):
    """GPU-only: sum over every token's experts of weight * row (expert order)."""
    out = torch.empty((weight.shape[0], y.shape[1]), dtype=y.dtype, device=y.device)
    _C.moe_combine(out, y, place, weight)
    return out


def quant_fp8_rows(x, src):
    """GPU-only: quant_fp8 of the rows src (int32) of x."""
    _require_ext()
    out = torch.empty(
        (src.shape[0], x.shape[1]), dtype=torch.float8_e4m3fn, device=x.device
    )
    scale = torch.empty(src.shape[0], dtype=torch.float32, device=x.device)
    _C.quant_fp8_rows(out, scale, x, src)
    return out, scale


def moe_mlp(x, router, top_k: int, gate_up, down, gate_up_scale=None, down_scale=None,
            gelu: bool = False):
    """GPU-only: sparse mixture of gated experts. x [T, H], router [E, H] (both
    bf16), gate_up [E, 2I, H] and down [E, H, I] in bf16, or fp8 with scales per
    output column (x is then quantized once, every expert's activations once).
    Router scores, weights and the sum over a token's experts are fp32."""
    weight, begin, src, place = moe_route(x, router, top_k)
    n = src.shape[0]
    h = torch.empty((n, gate_up.shape[1]), dtype=torch.bfloat16, device=x.device)
    y = torch.empty((n, x.shape[1]), dtype=torch.bfloat16, device=x.device)
    if gate_up_scale is not None:
        _C.skinny_experts(h, *_with_scale(quant_fp8(x), gate_up, gate_up_scale), begin, src)
        _C.skinny_experts(y, *_with_scale(silu_and_mul_fp8(h), down, down_scale), begin, None)
    else:
        _C.skinny_experts(h, x, gate_up, None, None, begin, src)
        a = gelu_and_mul(h) if gelu else silu_and_mul(h)
        _C.skinny_experts(y, a, down, None, None, begin, None)
    return moe_combine(y, place, weight)


def grouped_linear_takes(x, w) -> bool:
    """Whether grouped_linear multiplies rows like x by w [E, N, K] of x's type."""
    es = x.element_size()
    return (
        x.is_cuda
        and _C is not None
        and x.dtype == w.dtype
        and x.dtype in (torch.bfloat16, torch.float8_e4m3fn)
        and x.stride(1) == w.stride(2) == 1
        and w.shape[2] * es % 128 == 0
        and w.shape[2] * es < 2**23
        and w.shape[1] % 4 == 0
        and 0 < w.shape[0] < 65536
        and x.stride(0) * es % 16 == w.stride(0) * es % 16 == w.stride(1) * es % 16 == 0
        and x.stride(0) >= w.shape[2] <= w.stride(1)
        and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))
        and aligned(x, w)
    )


def grouped_linear_better(n: int, w) -> bool:
    """Whether n rows of w's experts are better multiplied by grouped_linear than
    by a library product per expert. fp8: always (8 experts, 512 rows each, us,
    grouped / library: 28672 x 4096 539/686, 4096 x 14336 284/474, without the look at
    the routing from the host). bf16: unless every expert's product fills the chip
    by itself (28672 x 4096 64 rows 364/431, 256 rows 576/596, 1024 rows 1666/1664, 2048
    rows 3233/2907; 12800 x 4096 2048 rows 2858/2730; 4096 x 14336 512 rows 540/803, 2048
    rows 1781/2260; 3584 x 2048 1024 rows 121/193, 2048 rows 249/275, 4096 rows
    467/388), or is short beside the look at the routing and the calls (a layer of 4
    of 1280 x 768 and 768 x 640, 3772 rows each 132/302)."""
    mean, N = n / w.shape[0], w.shape[1]
    return w.element_size() == 1 or mean <= 1024 or mean <= 3072 and N <= 8192 or (
        mean * N < 120 * 2**16
    )


def grouped_linear(x, w, bounds, src=None, scales=None, square=None, act=0):
    """GPU-only: rows of x [*, K] in expert order times their expert's matrix,
    w [E, N, K] (any strides of e and n), all experts in one launch. bounds int32:
    the experts' row counts [E] or offsets [E + 1]; src int32: the rows of x
    (all, in order). fp8 x and w: scales = (fp32 per row of x, [E, N]). square
    (fp32 per row): relu(product)^2 * square instead of the product. act: w is gate
    rows, then up rows (bf16); silu (1) or gelu (2) of gate times up [n, N / 2]."""
    _require_ext()
    n = x.shape[0] if src is None else src.shape[0]
    width = w.shape[1] // 2 if act else w.shape[1]
    y = torch.empty((n, width), dtype=torch.bfloat16, device=x.device)
    _C.grouped_linear(y, x, w, *(scales or (None, None)), bounds, src, square, act)
    return y


def _with_scale(quantized, weight, weight_scale):
    xq, xs = quantized
    return xq, weight, xs, weight_scale


def greedy_sample(logits):
    """The place of each row's largest value. On GPU a row in which none compares (all
    NaN) gives V, one behind the last; gumbel_sample and sample_with_logprobs do too."""
    if logits.is_cuda:
        _require_ext()
        out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
        _C.greedy_sample(out, logits)
        return out
    return ref.greedy_sample(logits)


def gumbel_sample(logits, temperature, seeds, step: int):
    if logits.is_cuda:
        _require_ext()
        out = torch.empty(logits.shape[0], dtype=torch.int64, device=logits.device)
        _C.gumbel_sample(out, logits, temperature, seeds, step)
        return out
    return ref.gumbel_sample(logits, temperature, seeds, step)


def fill_rows(out, rows) -> None:
    """out [R, C] int32 on the host: row i takes the list rows[i], zeros elsewhere (40
    lists of 30 cost numpy 50 us, this 5)."""
    if _C is not None:
        _C.fill_rows(out, rows)
        return
    out.zero_()
    for i, row in enumerate(rows):
        out[i, : len(row)] = torch.tensor(row, dtype=torch.int32)


def sample_with_logprobs(logits, temperature=None, seeds=None, step: int = 0):
    """(tokens [S], log-probabilities [S]) as one block of bytes on the logits' device,
    int64 then fp32 (sampled_to_host): greedy_sample, or with temperature and seeds
    gumbel_sample, and the tokens' logit - logsumexp(row). On GPU both come from one
    pass over the logits."""
    S = logits.shape[0]
    block = torch.empty(12 * S, dtype=torch.uint8, device=logits.device)
    tokens, logprobs = block[: 8 * S].view(torch.int64), block[8 * S :].view(torch.float32)
    if logits.is_cuda:
        _require_ext()
        if temperature is None:
            _C.greedy_sample(tokens, logits, logprobs)
        else:
            _C.gumbel_sample(tokens, logits, temperature, seeds, step, logprobs)
        return block
    if temperature is None:
        tokens.copy_(ref.greedy_sample(logits))
    else:
        tokens.copy_(ref.gumbel_sample(logits, temperature, seeds, step))
    chosen = logits.gather(1, tokens.view(-1, 1)).squeeze(1)
    logprobs.copy_(chosen - torch.logsumexp(logits, dim=-1))
    return block


def sampled_to_host(block):
    """The lists of a sample_with_logprobs block, in one copy."""
    host = block.cpu()
    S = host.numel() // 12
    return host[: 8 * S].view(torch.int64).tolist(), host[8 * S :].view(torch.float32).tolist()


def nucleus_stats(logits, temps):
    """Per-row (max, sum exp((x-max)/t)) for rejection nucleus sampling."""
    if logits.is_cuda:
        _require_ext()
        S = logits.shape[0]
        m = torch.empty(S, dtype=torch.float32, device=logits.device)
        z = torch.empty_like(m)
        _C.nucleus_stats(m, z, logits, temps)
        return m, z
    t = temps.clamp_min(1e-6).unsqueeze(1)
    m = logits.max(dim=-1).values
    z = torch.exp((logits - m.unsqueeze(1)) / t).sum(-1)
    return m, z


def nucleus_accept(logits, cand, m, z, temps, top_ps, top_ks):
    """uint8 mask: sampled token lies in the top-p/top-k nucleus
    (probability mass strictly above it < top_p, rank < top_k);
    greedy rows always accept, and on GPU a candidate outside the
    vocabulary (see greedy_sample) never does in the others."""
    if logits.is_cuda:
        _require_ext()
        ok = torch.empty(logits.shape[0], dtype=torch.uint8,
                         device=logits.device)
        _C.nucleus_accept(ok, logits, cand, m, z, temps, top_ps, top_ks)
        return ok
    t = temps.clamp_min(1e-6).unsqueeze(1)
    lt = logits.gather(1, cand.view(-1, 1))
    above = logits > lt
    mass = (torch.exp((logits - m.unsqueeze(1)) / t) * above).sum(-1) / z
    cnt = above.sum(-1)
    ok = (mass < top_ps) & ((top_ks <= 0) | (cnt < top_ks)) | (temps <= 0)
    return ok.to(torch.uint8)
