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


def paged_attention_decode(
    q, k_cache, v_cache, block_tables, seq_lens, scale: float, out=None,
    window: int = 0, softcap: float = 0.0,
):
    """q may be a row-strided view (fused qkv output); out must be
    contiguous (allocated here if not supplied). window > 0 enables
    sliding-window attention (Mistral/Gemma2 style: keys in
    (pos-window, pos])."""
    if q.is_cuda:
        _require_ext()
        if out is None:
            out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        _C.paged_attention_decode(
            out, q, k_cache, v_cache, block_tables, seq_lens, scale, window,
            softcap, None
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


def paged_attention_decode_fp8(
    q, k_cache, v_cache, block_tables, seq_lens, scale: float, window: int = 0,
    softcap: float = 0.0,
):
    """quant_fp8 of paged_attention_decode's rows [B, n_q * hd]. On GPU the merge of
    a row's splits converts them, where there is more than one."""
    B, n_q, hd = q.shape
    if not q.is_cuda or n_q > 128 or B == 0 or (
        _C.paged_decode_splits(B, k_cache.shape[1], hd, block_tables.shape[1]) == 1
    ):
        out = paged_attention_decode(q, k_cache, v_cache, block_tables, seq_lens, scale,
                                     window=window, softcap=softcap)
        return quant_fp8(out.view(B, n_q * hd))
    out = torch.empty((B, n_q * hd), dtype=torch.float8_e4m3fn, device=q.device)
    out_scale = torch.empty(B, dtype=torch.float32, device=q.device)
    _C.paged_attention_decode(out, q, k_cache, v_cache, block_tables, seq_lens, scale,
                              window, softcap, out_scale)
    return out, out_scale


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
    library / this: bf16 4096 -> 4096 8 rows 18.9 / 13.5, 96 rows 25.3 / 19.3;
    14336 -> 4096 8 rows 30.4 / 31.0, 40 rows 39.4 / 32.1; 4096 -> 6144 8 rows 18.4
    / 16.2 (rotation), 64 rows 20.4 / 21.2; 8192 -> 8192 34.7 / 41.4; 8192 -> 1024
    8 rows 14.6 / 12.3, 40 rows 15.1 / 17.1. fp8 4096 -> 4096 16 rows 15.8 / 13.3,
    64 rows 16.4 / 18.3; 14336 -> 4096 40 rows 25.1 / 22.8; 8192 -> 8192 8 rows
    47.5 / 26.6, 16 rows 20.6 / 27.2; 512 -> 4096 8.2 / 8.8. Over 3576 and 1656
    products of 512 to 28672 columns and rows with either reader the chosen ones
    take 0.72 and 0.80 of the library's time, the worst 1.2.
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


def _streams_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether the weight-streaming product beats the library's where it has to
    add its parts itself. Few rows and a width that fills the chip uncut (us,
    weights out of cache, library / this, 8 rows): bf16 4096 -> 28672 59.9 / 47.6,
    2304 -> 18432 50.8 / 25.2, 2048 -> 32256 34.5 / 31.4, 4096 -> 65536 123 / 107,
    but 4096 -> 16384 33.4 / 34.8, 8192 -> 24576 83.8 / 91.8, 6144 -> 24576 at 16
    rows 68.5 / 73.8; fp8 4096 -> 16384 27.9 / 20.3, 4096 -> 28672 33.8 / 28.0,
    8192 -> 30720 65 / 58; beyond two passes of workgroups over the chip only
    whole passes (8192 -> 36864 fp8 72 / 81), and not for rows under 256 bytes (128
    -> 65536 fp8 5.6 / 6.7). At 32 rows 53.5 / 53.4 and 21 / 30, at 128256 columns
    192 / 198. Very long rows, which the library does not cut: 32256 -> 2048 83 /
    38 at 8 rows, 127 / 60 at 96; it does at 16384 (-> 1024 20.4 / 19.4 at 8 rows,
    21.0 / 28.7 at 48; fp8 20.2 / 12.9, 20.1 / 21.4 at 96)."""
    if K >= 8 * N and K >= 16384:
        return K > 16384 or M <= (64 if fp8 else 32)
    if M > 16 or N > 65536 or (N > 32768 and N % 16384) or K * (1 if fp8 else 2) < 256:
        return False
    if fp8:
        return N >= 16384 and K <= 8192
    return N >= 16384 and K <= 1024 or N > 16384 and K <= (6144 if M <= 8 else 4096)


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


def _tiled_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether the tiled product (csrc/tiled_gemm.h) beats the library's. fp8: from
    97 rows on, unless K is short, where the stores count (us, weights out of
    cache, library / this: 16384 x 512 8192 rows 104 / 127, 1024 x 1024 4.8 / 5.8) or
    so long that the tiles of few columns leave CUs idle while few rows are
    multiplied (4096 x 14336 256 rows 34 / 49, 2304 x 9216 160 rows 16 / 22; 640 rows
    72 / 63 and 29 / 28). Over 137 others (97 to 8192 rows, 2048 to 32000 columns) it
    takes 0.87 of the library's time, 1.06 at worst. Logits of few rows: 128256 x
    4096 fp8 40 rows 129 / 107, 96 rows 121 / 118, bf16 40 rows 203 / 192, 160
    rows 246 / 213, 384 rows 437 / 339, 1024 rows 853 / 838; 57344 x 8192 fp8 40 rows
    121 / 103. Other bf16 products stay (28672 x 4096 2048 rows 333 / 391)."""
    if N >= 49152 and K >= 2048:
        return M > 16 and (fp8 or M <= 1024 and N >= 98304)
    return fp8 and M > 96 and K >= 2048 and (K <= 2 * N or M > 512)


def _tiled_linear(x, weight, x_scale=None, w_scale=None, out=None, act=0):
    if out is None:
        out = torch.empty(
            (x.shape[0], weight.shape[0] // (2 if act else 1)), dtype=torch.bfloat16,
            device=x.device,
        )
    _C.tiled_linear(out, x, weight, x_scale, w_scale, act)
    return out


def tiled_gated(x, weight, x_scale=None, w_scale=None, gelu=False):
    """silu_and_mul (gelu: gelu_and_mul) of x weight^T (weight: gate rows, then up
    rows) in one launch, the activation in fp32 and rounded once; None where the
    product is not a tiled one or two launches are faster. fp8 (silu): where the
    product is tiled anyway; bf16: up to 512 rows, with K up to 2560 up to 1024 (us,
    library and activation / this: 28672 x 4096 128 rows 58.0 / 54.9, 384 rows 92 /
    89, 640 rows 150 / 160, 2048 rows 381 / 408; 22016 x 4096 640 rows 125 / 121, 1024
    rows 173 / 191; 18432 x 2304 gelu 384 rows 45.9 / 41.4, 1024 rows 102 / 94, 2048
    rows 172 / 181, 5376 rows 399 / 382 alone but 379 / 385 in a model)."""
    (M, K), N = x.shape, weight.shape[0]
    if x_scale is not None:
        better = M > 96 and not gelu and _tiled_better(M, N, K, fp8=True)
    else:
        better = 96 < M and N >= 8192 and K >= 2048 and (
            M <= 512 or K <= 2560 and M <= 1024
        )
    if not (
        better and weight.dim() == 2 and N * weight.stride(0) * weight.element_size() < 2**31
        and _tiled_operands(x, weight)
    ):
        return None
    return _tiled_linear(x, weight, x_scale, w_scale, act=2 if gelu else 1)


#: Products of more rows are not handed on as sums: whole ones fill the chip.
MAX_SUM_ROWS = 2048


@functools.lru_cache(maxsize=4096)
def tiled_sums_better(M: int, N: int, K: int, fp8: bool) -> bool:
    """Whether a product of more than 96 rows as ProductSums of a tiled product
    that is cut along K, and the norm or rotation that adds them, beat the product
    as a whole and its reader: where its tiles alone leave CUs idle. By the costs
    of both (csrc/tiled_gemm.hip) and 3.5 us that a reader of few rows takes longer.
    Over 50 products (128 to 1024 rows, 1024 to 10240 columns, K 1024 to 28672) of each
    type, against the tiled product in fp8 and the library in bf16, with either
    reader, the chosen ones gain 1.5 and 1.35 in the mean, 0.93 at worst (us with the
    norm: 4096 x 14336 128 rows fp8 51 / 26, bf16 76 / 35; 512 rows 53 / 49, 92 / 70; 1024
    rows bf16 139 / 116; 4096 x 4096 128 rows bf16 28 / 19, fp8 15.5 / 16.7: whole)."""
    es = 1 if fp8 else 2
    if _C is None or not 96 < M <= MAX_SUM_ROWS or N > 16384 or K * es % 128:
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
    Else the library's product and reader / this: fp8 3072 x 8192 40 rows 17.1 / 16.0
    (rotation 16.9 / 17.0), 96 rows 25.4 / 17.8; 8192 x 28672 40 rows 74 / 52; 8192 x
    8192 40 rows 22.6 / 24.7; bf16 6144 x 4096 40 rows 20.4 / 17.9, 96 rows 25.9 / 20.7;
    10240 x 8192 24 rows 41.1 / 40.7, 96 rows 54.9 / 42.9; 2304 x 2048 80 rows 12.0 /
    12.6. Over 78 products with either reader a step of these rows takes 0.93 (fp8) and
    0.92 (bf16) of the time that it took with the streaming product alone."""
    if sums:
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


def tiled_sums(x, weight, x_scale=None, w_scale=None):
    """x weight^T as ProductSums of the tiled product, cut along K so that it
    fills the chip, or None for operands that it does not take."""
    if not _tiled_operands(x, weight):
        return None
    return ProductSums(_C.tiled_sums(x, weight), x_scale, w_scale)


def sums_for_reader(x, weight, x_scale=None, w_scale=None, rope=False, eager=False):
    """x weight^T (fp8 with the scales of both) as ProductSums where that and the
    norm, or (rope) the rotation, that reads it are the fastest form, or None: the
    product as a whole. eager: see sums_better."""
    M, (N, K), fp8 = x.shape[0], weight.shape, x_scale is not None
    if M > 96:
        better = tiled_sums_better(M, N, K, fp8)
        return tiled_sums(x, weight, x_scale, w_scale) if better else None
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
        and _skinny_operands(xq, weight)
        and (out is None or out.is_contiguous())
    ):
        if out is None:
            out = torch.empty(
                (xq.shape[0], weight.shape[0]), dtype=torch.bfloat16, device=xq.device
            )
        _C.skinny_linear(out, xq, weight, x_scale.reshape(-1), w_scale.reshape(-1), bias)
        return out
    if (
        bias is None
        and _tiled_better(xq.shape[0], *weight.shape, fp8=True)
        and _tiled_operands(xq, weight)
        and (out is None or out.is_contiguous() and out.dtype == torch.bfloat16)
    ):
        return _tiled_linear(xq, weight, x_scale.reshape(-1), w_scale.reshape(-1), out)
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
    """hidden = x + residual in bf16 and its norm; returns (norm, hidden). x may be
    ProductSums or a BranchNorm (then its norm is added). On GPU one launch, with the
    bits of rmsnorm, the addition and rmsnorm after one another."""
    w1 = None
    if isinstance(x, BranchNorm):
        if x.eps == eps and _norm_add_norm_takes(x.x, residual, x.weight, weight):
            x, w1 = x.x, x.weight
        else:
            x = rmsnorm(x.x, x.weight, x.eps)
    if not (w1 is not None or _norm_add_norm_takes(x, residual, None, weight)):
        if isinstance(x, ProductSums):
            raise RuntimeError("a product's sums beside a residual that is not dense bf16")
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
    467/388)."""
    mean = n / w.shape[0]
    return w.element_size() == 1 or mean <= 1024 or mean <= 3072 and w.shape[1] <= 8192


def grouped_linear(x, w, bounds, src=None, scales=None, square=None, act=0):
    """GPU-only: rows of x [*, K] in expert order times their expert's matrix,
    w [E, N, K] (any strides of e and n), all experts in one launch. bounds int32:
    the experts' row counts [E] or offsets [E + 1]; src int32: the rows of x
    (all, in order). fp8 x and w: scales = (fp32 per row of x, [E, N]). square
    (fp32 per row): relu(product)^2 * square instead of the product. act: w is gate
    rows, then up rows; silu (1) or, in bf16, gelu (2) of gate times up [n, N / 2]."""
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
    greedy rows always accept."""
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
