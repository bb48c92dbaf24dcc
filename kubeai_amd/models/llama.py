"""Llama-family decoder for the kubeai_amd engine.

MI355X-first execution model (one process per GPU):
  - token-packed forward ([T, H], no padding) over the ForwardBatch;
  - products (qkv/o/gate_up/down/lm_head) go through ops.linear: the
    weight-streaming or the tiled kernel where they are the faster ones, as
    sums that the next norm or rotation adds or with the activation behind
    them, hipBLASLt for the rest; every other hot op (rmsnorm, rope, cache
    write, paged attention) is a hand-written gfx950 kernel via kubeai_amd.ops;
  - KV cache is paged [num_blocks, n_kv, block_size, head_dim] bf16, owned by
    the runner and passed in.

Reference parity: this is the in-house engine the reference delegates to
vLLM pods for; no reference code exists for it.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F

from kubeai_amd import ops
from kubeai_amd.engine.batch import ForwardBatch
from .config import ModelArchConfig


class EngineLinear(nn.Linear):
    """nn.Linear routed through ops.linear. Bias (Qwen2 qkv) is added outside
    the product."""

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        y = ops.linear(x, self.weight)
        if self.bias is not None:
            y = y + self.bias
        return y

    def sums(self, x: torch.Tensor, rope: bool = False, eager: bool = False):
        """The product as ops.ProductSums, for a norm or (rope) the rotation, or
        None (library product, bias)."""
        if self.bias is not None:
            return None
        return ops.sums_for_reader(x, self.weight, rope=rope, eager=eager)


_EVERY_MODULES_HOOKS = torch.nn.modules.module._global_forward_hooks
_EVERY_MODULES_PRE_HOOKS = torch.nn.modules.module._global_forward_pre_hooks


def _hooked(module: nn.Module) -> bool:
    """Whether someone waits for the module's call and its tensors, or has put a
    forward of their own into it."""
    return bool(
        "forward" in module.__dict__ or module._forward_hooks or module._forward_pre_hooks
        or _EVERY_MODULES_HOOKS or _EVERY_MODULES_PRE_HOOKS
    )


def _project(linear, x, as_sums: bool, fb: ForwardBatch | None, rope: bool = False):
    """linear(x), x a tensor or an (fp8 rows, scales) pair. as_sums: what reads
    the result, a norm or (rope) the rotation, takes ops.ProductSums, so it may
    be that. Steps with prompt portions or adapters are never recorded in a graph."""
    eager = fb is not None and (fb.n_prefill > 0 or fb.lora_ids is not None)
    if isinstance(x, tuple):
        sums = getattr(linear, "sums_quantized", None) if as_sums else None
        y = sums(*x, rope, eager) if sums is not None else None
        return linear.forward_quantized(*x) if y is None else y
    y = None
    if as_sums and type(linear) is EngineLinear and not _hooked(linear):
        y = linear.sums(x, rope, eager)
    return linear(x) if y is None else y


def _project_adapted(linear, x, as_sums: bool, fb, lm, layer_idx, target, rope=False):
    """_project with the adapters' products of x added: to the first part of the
    sums, where the adapters go in one batch."""
    batch = None
    if as_sums and isinstance(linear, nn.Linear):
        batch = lm.batch(layer_idx, target, x, fb.lora_ids, linear.out_features)
    y = _project(linear, x, batch is not None, fb, rope)
    if isinstance(y, ops.ProductSums):
        lm.apply_batch(batch, x, y.part[0], fb.lora_ids)
    else:
        lm.apply(layer_idx, target, x, y, fb.lora_ids)
    return y


def _call(module, *args, **own):
    return module(*args)


def _branch(module, *args, **own):
    """The attention or feed-forward module's result, ops.ProductSums where it
    is one that can give them and nobody else sees what it returns. own: what
    only the modules of this file take."""
    if type(module) in (Attention, MLP, MoEMLP) and not _hooked(module):
        return module(*args, **own, as_sums=True)
    return module(*args)


def _rms_head(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """Per-head RMSNorm over the last dim (gemma3 qk-norm).

    On GPU this routes through the rmsnorm HIP kernel on a [T*heads, hd]
    view (one copy + one kernel instead of ~6 eager elementwise ops —
    these run inside the decode hipGraph every layer)."""
    if x.is_cuda and x.dtype == torch.bfloat16:
        flat = x.contiguous().view(-1, x.shape[-1])
        return ops.rmsnorm(flat, w, eps).view(x.shape)
    xf = x.float()
    xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    return (xf * w.float()).to(x.dtype)


class Attention(nn.Module):
    def __init__(self, cfg: ModelArchConfig, layer_idx: int):
        super().__init__()
        self.layer_idx = layer_idx
        self.n_q = cfg.num_attention_heads
        self.n_kv = cfg.num_key_value_heads
        self.hd = cfg.head_dim
        # per-layer window: gemma2 interleaves windowed ("even" layers)
        # and full-causal attention; gemma3 makes every Nth layer GLOBAL
        # (others windowed, local rope base); mistral windows every layer
        if cfg.global_layer_interval > 0:
            self.is_global = (layer_idx + 1) % cfg.global_layer_interval == 0
            use_win = not self.is_global
        else:
            self.is_global = True
            use_win = (
                cfg.sliding_window_pattern != "even" or layer_idx % 2 == 0
            )
        self.window = (cfg.sliding_window or 0) if use_win else 0
        self.qk_norm = cfg.qk_norm
        if cfg.qk_norm:
            self.q_norm = nn.Parameter(torch.ones(cfg.head_dim))
            self.k_norm = nn.Parameter(torch.ones(cfg.head_dim))
        self.norm_eps = cfg.rms_norm_eps
        self.softcap = cfg.attn_logit_softcap or 0.0
        self.scale = (
            cfg.attention_multiplier
            or 1.0 / math.sqrt(cfg.query_pre_attn_scalar or self.hd)
        )
        q_size = self.n_q * self.hd
        kv_size = self.n_kv * self.hd
        self.qkv_proj = EngineLinear(
            cfg.hidden_size, q_size + 2 * kv_size, bias=cfg.attention_bias
        )
        self.o_proj = EngineLinear(q_size, cfg.hidden_size, bias=False)

    def forward(
        self,
        x: torch.Tensor,  # [T, H]
        fb: ForwardBatch,
        kv_cache: tuple[torch.Tensor, torch.Tensor],
        cos_sin: torch.Tensor,
        as_sums: bool = False,
    ) -> torch.Tensor:
        """as_sums: the caller takes the result as ops.ProductSums too."""
        fp8_in = isinstance(x, tuple)  # (fp8 tensor, row scales) from a
        # fused producer kernel (DecoderLayer fp8 path)
        k_cache, v_cache = kv_cache
        T = (x[0] if fp8_in else x).shape[0]
        lm = None if fp8_in else getattr(self, "_lora_manager", None)
        lora_live = lm is not None and lm.active and fb.lora_ids is not None
        qkv_sums = (
            T <= ops.MAX_SUM_ROWS and not self.qk_norm
            and ops.rope_takes_sums(k_cache, v_cache)
        )
        if lora_live:
            qkv = _project_adapted(
                self.qkv_proj, x, qkv_sums, fb, lm, self.layer_idx, "qkv", rope=True
            )
        else:
            qkv = _project(self.qkv_proj, x, qkv_sums, fb, rope=True)
        if isinstance(cos_sin, tuple):
            # (global, local) caches — gemma3 dual rope bases
            cos_sin = cos_sin[0] if self.is_global else cos_sin[1]
        nd = fb.n_decode
        plan = ops.decode_plan(
            fb.decode_plans, fb.decode_seq_lens, fb.decode_block_tables, k_cache, self.window,
            alone=fb.n_prefill == 0,
        ) if nd > 0 else None
        if nd == T and fb.n_prefill == 0 and ops.decode_takes_sums(
            qkv, self.n_q, cos_sin, k_cache, v_cache
        ):
            out = ops.paged_attention_decode_sums(
                qkv, self.n_q, fb.positions, cos_sin, fb.slot_mapping, k_cache, v_cache,
                fb.decode_block_tables, fb.decode_seq_lens, self.scale,
                window=self.window, softcap=self.softcap, plan=plan, fp8=fp8_in,
            )
            if not fp8_in:
                out = out.view(T, -1)
            return self._out_proj(out, fb, lm if lora_live else None, as_sums)
        if self.qk_norm:
            # gemma3: per-head RMSNorm ((1+w) stored as w) before rope;
            # fp32 math, contiguous bf16 out. v follows to contiguous —
            # the cache-write kernel wants k/v with one shared row stride
            q, k, v = qkv.split(
                [self.n_q * self.hd, self.n_kv * self.hd, self.n_kv * self.hd],
                dim=-1,
            )
            q = _rms_head(
                q.unflatten(-1, (self.n_q, self.hd)), self.q_norm, self.norm_eps
            )
            k = _rms_head(
                k.unflatten(-1, (self.n_kv, self.hd)), self.k_norm, self.norm_eps
            )
            v = v.unflatten(-1, (self.n_kv, self.hd)).contiguous()
            q, k = ops.rope(q, k, fb.positions, cos_sin)
            ops.reshape_and_cache(k, v, k_cache, v_cache, fb.slot_mapping)
        else:
            q = ops.rope_and_cache(
                qkv, self.n_q, fb.positions, cos_sin, k_cache, v_cache,
                fb.slot_mapping,
            )

        if fp8_in and nd == T and fb.n_prefill == 0:
            return _project(
                self.o_proj,
                ops.paged_attention_decode_fp8(
                    q, k_cache, v_cache, fb.decode_block_tables, fb.decode_seq_lens,
                    self.scale, window=self.window, softcap=self.softcap, plan=plan,
                ),
                as_sums, fb,
            )
        if plan is not None and fb.n_prefill > 0 and ops.step_attention_takes(
            q, nd, k_cache, plan
        ):
            out = ops.paged_attention_step(
                q, nd, k_cache, v_cache, fb.decode_block_tables, fb.decode_seq_lens,
                fb.prefill_block_tables, fb.prefill_query_start_loc, fb.prefill_seq_lens,
                self.scale, window=self.window, softcap=self.softcap, plan=plan, fp8=fp8_in,
            )
            if fp8_in:
                return _project(self.o_proj, out, as_sums, fb)
            return self._out_proj(out.view(T, -1), fb, lm if lora_live else None, as_sums)
        out = torch.empty(
            (T, self.n_q, self.hd), dtype=q.dtype, device=q.device
        )
        if nd > 0:
            ops.paged_attention_decode(
                q[:nd],
                k_cache,
                v_cache,
                fb.decode_block_tables,
                fb.decode_seq_lens,
                self.scale,
                out=out[:nd],
                window=self.window,
                softcap=self.softcap,
                plan=plan,
            )
        if fb.n_prefill > 0:
            ops.paged_attention_prefill(
                q[nd:],
                k_cache,
                v_cache,
                fb.prefill_block_tables,
                fb.prefill_query_start_loc,
                fb.prefill_seq_lens,
                self.scale,
                out=out[nd:],
                window=self.window,
                softcap=self.softcap,
            )
        attn_flat = out.view(T, -1)
        if fp8_in:
            return _project(self.o_proj, ops.quant_fp8(attn_flat), as_sums, fb)
        return self._out_proj(attn_flat, fb, lm if lora_live else None, as_sums)

    def _out_proj(self, x, fb, lm, as_sums: bool):
        """lm: the adapters that are live in this step, or None."""
        if lm is not None:
            return _project_adapted(self.o_proj, x, as_sums, fb, lm, self.layer_idx, "o")
        return _project(self.o_proj, x, as_sums, fb)


class MLP(nn.Module):
    def __init__(self, cfg: ModelArchConfig, layer_idx: int | None = None):
        super().__init__()
        # layer_idx set only for the DENSE per-layer MLP: LoRA targets it
        # (MoE expert MLPs pass None — adapters stay attention-only there)
        self.layer_idx = layer_idx
        self.gate_up_proj = EngineLinear(
            cfg.hidden_size, 2 * cfg.intermediate_size, bias=False
        )
        self.down_proj = EngineLinear(cfg.intermediate_size, cfg.hidden_size, bias=False)
        self.gelu = cfg.hidden_act == "gelu_pytorch_tanh"

    def forward(
        self, x, fb: ForwardBatch | None = None, as_sums: bool = False
    ) -> torch.Tensor:
        """as_sums: the caller takes the result as ops.ProductSums too."""
        if isinstance(x, tuple):  # fused fp8 path (never active with LoRA)
            # (in the product's epilogue the activation would lie in bf16, or in
            # fp32 rows of gate and up's size, until a row's scale is known)
            h = self.gate_up_proj.forward_quantized(*x)
            return _project(self.down_proj, ops.silu_and_mul_fp8(h), as_sums, fb)
        lm = getattr(self, "_lora_manager", None)
        lora_live = (
            lm is not None and lm.active and fb is not None
            and fb.lora_ids is not None and self.layer_idx is not None
        )
        a = None
        if not (
            lora_live or x.dim() != 2
            or type(self.gate_up_proj) is not EngineLinear or _hooked(self.gate_up_proj)
            or self.gate_up_proj.bias is not None
        ):
            a = ops.gated(x, self.gate_up_proj.weight, gelu=self.gelu)
        if a is None:
            h = self.gate_up_proj(x)
            if lora_live:
                if not self.gelu:
                    a = lm.gated(self.layer_idx, x, h, fb.lora_ids)
                if a is None:
                    lm.apply(self.layer_idx, "gate_up", x, h, fb.lora_ids)
            if a is None:
                a = ops.gelu_and_mul(h) if self.gelu else ops.silu_and_mul(h)
        if lora_live:
            return _project_adapted(
                self.down_proj, a, as_sums, fb, lm, self.layer_idx, "down"
            )
        return _project(self.down_proj, a, as_sums, fb)


def _own_tensor(module: nn.Module, name: str):
    t = module._parameters.get(name)
    return module._buffers.get(name) if t is None else t


def _restack_after_load(module: "MoEMLP", _) -> None:
    module._restack()


class MoEMLP(nn.Module):
    """Mixtral-style sparse MoE block (token-level top-k routing).

    On GPU, small steps route on the device
    (csrc/moe.hip) and run all experts' rows in one weight-streaming product
    per projection (csrc/skinny_gemm.hip): shapes do not depend on the routing,
    so decode steps can be recorded in a graph, and every expert's weights are
    read once, for its own rows only. The experts' weights lie behind one
    another in one tensor for that; the modules' parameters are views of it.
    Larger steps sort the rows by expert on the device; a projection is one
    tiled product for all experts (csrc/tiled_gemm.h) or, where that is the
    slower one, the library's on each expert's slice, after one look at the
    experts' row counts."""

    #: one pass of 8 experts of 14336 x 4096, us, weight-streaming / tiled: fp8 128
    #: tokens 355/302, 256 405/325; bf16 643/557, 704/572; every expert's tokens
    #: asked for one after the other took 722 and 1159 at 128. (Streaming reads an
    #: expert's weights again for every 96 of its rows.) Up to 256 tokens any
    #: routing may be recorded in a graph, so no row counts come to the host.
    GROUPED_MAX_TOKENS = 256

    #: Above these the tiled product has the step where it takes both
    #: projections. us, streaming / tiled, tokens spread evenly (half of them
    #: alike): fp8 8 x 14336 x 4096 160 tokens 371/308 (428/343), 192 382/334
    #: (465/358), 256 405/325 (500/378); 8 x 7168 x 2048 160 129/120 (155/124), 192
    #: 131/121 (166/128); 16 x 6400 x 4096 160 302/288 (359/308), 192 316/290
    #: (348/309); 32 x 1408 x 2048, 4 a token, 160 112/111 (138/121), 192 118/112
    #: (141/123); 4 x 3584 x 1024 160 62/49 (77/50), 192 76/50 (84/57). bf16 8 x 14336 x
    #: 4096 224 681/565 (910/676), 256 704/572 (958/674); 8 x 7168 x 2048 224 215/201
    #: (282/211), 256 220/200 (304/210); 16 x 6400 x 4096 224 573/504 (659/550), 256
    #: 569/491 (721/523); 32 x 1408 x 2048 224 170/168 (204/182), 256 173/169
    #: (223/180). The lines are where the two met before experts' tiles went by the
    #: costs of one matrix. The tiled kernel is the faster one from fewer tokens on
    #: now, down to 128 at most of these sizes; the lines have not been moved since.
    #: (The kernels need not round alike, and in a routed model that can move a token
    #: whose scores all but tie.)
    TILED_ABOVE_FP8 = 160
    TILED_ABOVE_BF16 = 224

    def __init__(self, cfg: ModelArchConfig):
        super().__init__()
        self.n_experts = cfg.num_local_experts
        self.top_k = cfg.num_experts_per_tok
        self.gate = nn.Linear(cfg.hidden_size, self.n_experts, bias=False)
        with torch.device("meta"):  # their weights are views, made below
            self.experts = nn.ModuleList([MLP(cfg) for _ in range(self.n_experts)])
        self.gelu = cfg.hidden_act == "gelu_pytorch_tanh"
        self._stacks = {
            (proj, "weight"): torch.empty(
                (self.n_experts,) + getattr(self.experts[0], proj).weight.shape
            )
            for proj in ("gate_up_proj", "down_proj")
        }
        for e, expert in enumerate(self.experts):
            for proj in ("gate_up_proj", "down_proj"):
                lin = getattr(expert, proj)
                lin.weight = nn.Parameter(self._stacks[proj, "weight"][e])
                lin.reset_parameters()
        self.register_load_state_dict_post_hook(_restack_after_load)

    def stack_experts(self) -> None:
        """Put the experts' weights (and fp8 scales) behind one another and
        leave views of them in the modules. Called again when the modules
        or their tensors have been replaced (fp8 conversion)."""
        self._stacks = {}
        for proj in ("gate_up_proj", "down_proj"):
            mods = [getattr(e, proj) for e in self.experts]
            if any(getattr(m, "bias", None) is not None for m in mods):
                self._stacks = {}
                return
            for name in ("weight_fp8", "weight_scale", "weight"):
                parts = [_own_tensor(m, name) for m in mods]
                if any(t is None for t in parts) or len(
                    {(t.shape, t.dtype, t.device) for t in parts}
                ) != 1:
                    continue
                with torch.inference_mode(False), torch.no_grad():
                    stack = torch.stack(parts)
                self._stacks[proj, name] = stack
                for m, t, v in zip(mods, parts, stack):
                    if isinstance(t, nn.Parameter):
                        t.data = v
                    else:
                        m._buffers[name] = v
                del parts, t

    def _stack(self, proj: str, name: str):
        """The stacked tensor, or None where a module's own tensor has been
        moved out of it since (it is let go then)."""
        stack = self._stacks.get((proj, name))
        if stack is None:
            return None
        at, step = stack.data_ptr(), stack.stride(0) * stack.element_size()
        for e in self.experts:
            t = _own_tensor(getattr(e, proj), name)
            if t is None or t.data_ptr() != at or t.shape != stack.shape[1:]:
                self._stacks.pop((proj, name), None)
                return None
            at += step
        return stack

    # The stacks go where the modules' tensors go: to another device or type,
    # into a copy or a pickle, to the tensors that a state dict assigns.
    def _restack(self) -> None:
        kinds = list(self._stacks)
        if any(self._stack(*k) is None for k in kinds):
            self.stack_experts()

    def _apply(self, fn, recurse=True):
        super()._apply(fn, recurse)
        self._restack()
        return self

    def __getstate__(self):
        return {**self.__dict__, "_stacks": {}}

    def __setstate__(self, state):
        super().__setstate__(state)
        self.stack_experts()

    def _own_experts(self) -> bool:
        """Whether the experts are the modules made here (or their fp8 forms) and
        nobody waits for their calls: their weights may be used beside them."""
        for e in self.experts:
            if type(e) is not MLP or _hooked(e):
                return False
            for proj in ("gate_up_proj", "down_proj"):
                lin = e._modules[proj]
                if _hooked(lin) or "forward_quantized" in lin.__dict__ or not (
                    type(lin) is EngineLinear or "weight_fp8" in lin._buffers
                ):
                    return False
        return True

    def _routes(self) -> bool:
        """Whether csrc/moe.hip takes the routing of such rows as _on_device asks for."""
        gate = self.gate.weight
        return (
            gate.dtype == torch.bfloat16
            and gate.shape[1] % 8 == 0
            and gate.is_contiguous()
            and ops.aligned(gate)
            and self.n_experts <= 32
            and self.top_k <= min(8, self.n_experts)
            and self._own_experts()
        )

    def sorts_here(self) -> bool:
        """Whether steps of more than GROUPED_MAX_TOKENS have their routing and, for
        all experts, both projections from kernels here, whatever their size. (In bf16
        that depends on the rows.)"""
        if not self._routes():
            return False
        for proj in ("gate_up_proj", "down_proj"):
            w = self._stack(proj, "weight_fp8")
            if w is None or self._stack(proj, "weight_scale") is None or (
                not ops.grouped_linear_takes(w[0], w)
            ):
                return False
        return True

    def _on_device(self, x: torch.Tensor) -> bool:
        """Whether csrc/moe.hip takes the routing of x."""
        return (
            x.is_cuda
            and x.dtype == torch.bfloat16
            and x.is_contiguous()
            and x.shape[0] >= 1
            and x.stride(0) == x.shape[1]  # (of a single row it may be anything)
            and not torch.is_grad_enabled()
            and ops.aligned(x)
            and self._routes()
        )

    def _sorted(self, x: torch.Tensor) -> torch.Tensor:
        """Rows in expert order, one product per projection for all experts, or
        the library's for one after the other."""
        weight, begin, src, place = ops.moe_route(x, self.gate.weight, self.top_k)
        n = src.shape[0]
        first = self.experts[0]
        fp8 = hasattr(first.gate_up_proj, "forward_quantized")
        ends = None

        def products(rows, proj, width, src=None, act=0):
            """act: of gate and up rows; the result has half the width then, or
            the whole where the activation is still to be done."""
            nonlocal ends
            rows, scale = rows if fp8 else (rows, None)
            w = self._stack(proj, "weight_fp8" if fp8 else "weight")
            ws = self._stack(proj, "weight_scale") if fp8 else None
            if (
                w is not None and (ws is not None) == fp8
                and ops.grouped_linear_takes(rows, w) and ops.grouped_linear_better(n, w)
            ):
                if w.shape[1] % 16 or w.shape[1] * w.stride(1) * w.element_size() >= 2**31:
                    act = 0
                return ops.grouped_linear(
                    rows, w, begin, src=src, scales=(scale, ws) if fp8 else None,
                    act=act,
                )
            if src is not None:
                rows = rows.index_select(0, src)
            if ends is None:
                ends = begin.tolist()
            y = torch.empty((n, width), dtype=x.dtype, device=x.device)
            for e, expert in enumerate(self.experts):
                lo, hi = ends[e], ends[e + 1]
                if lo == hi:
                    continue
                lin = getattr(expert, proj)
                if fp8:
                    ops.linear_fp8(
                        rows[lo:hi], scale[lo:hi], lin.weight_fp8,
                        lin.weight_scale, lin.bias, out=y[lo:hi],
                    )
                else:
                    torch.mm(rows[lo:hi], lin.weight.t(), out=y[lo:hi])
            return y

        width = 2 * first.down_proj.in_features
        # Steps that the weight-streaming product may have as well round gate and up
        # as it does, before the activation; larger ones have it in the tiled product,
        # which saves these rows' way to memory and back.
        # (not in fp8: the activation stays in fp32 until it is converted)
        if fp8:
            h = products(ops.quant_fp8_rows(x, src), "gate_up_proj", width)
            a = ops.silu_and_mul_fp8(h)
        else:
            fused = x.shape[0] > self.GROUPED_MAX_TOKENS
            act = 0 if not fused else 2 if self.gelu else 1
            a = products(x, "gate_up_proj", width, src, act)
            if a.shape[1] == width:
                a = ops.gelu_and_mul(a) if self.gelu else ops.silu_and_mul(a)
        return ops.moe_combine(products(a, "down_proj", x.shape[1]), place, weight)

    def _tiled_has(self, tokens: int) -> bool:
        """Whether a step of up to GROUPED_MAX_TOKENS is the tiled product's."""
        fp8 = ("down_proj", "weight_fp8") in self._stacks
        if tokens <= (self.TILED_ABOVE_FP8 if fp8 else self.TILED_ABOVE_BF16):
            return False
        for proj in ("gate_up_proj", "down_proj"):
            w = self._stack(proj, "weight_fp8" if fp8 else "weight")
            if (
                w is None or (fp8 and self._stack(proj, "weight_scale") is None)
                or w.shape[2] * w.element_size() % 128 or w.shape[1] % 16
                or not ops.aligned(w)
                or not ops.grouped_linear_better(tokens * self.top_k, w)
            ):
                return False
        return not (fp8 and self.gelu)

    def _grouped(self, x: torch.Tensor):
        """All experts' rows at once; None where the kernels do not take it."""
        if not (self._on_device(x) and x.shape[0] <= self.GROUPED_MAX_TOKENS):
            return None
        fp8 = ("down_proj", "weight_fp8") in self._stacks
        name = "weight_fp8" if fp8 else "weight"
        gu, dn = self._stack("gate_up_proj", name), self._stack("down_proj", name)
        if gu is None or dn is None or (
            gu.shape[2] * gu.element_size() % 64 or dn.shape[2] * dn.element_size() % 64
            or gu.shape[1] % 16 or dn.shape[1] % 8
        ):
            return None
        if not fp8:
            return ops.moe_mlp(x, self.gate.weight, self.top_k, gu, dn, gelu=self.gelu)
        gs = self._stack("gate_up_proj", "weight_scale")
        ds = self._stack("down_proj", "weight_scale")
        if gs is None or ds is None or self.gelu:
            return None
        return ops.moe_mlp(x, self.gate.weight, self.top_k, gu, dn, gs, ds)

    def forward(
        self, x: torch.Tensor, fb: ForwardBatch | None = None, as_sums: bool = False
    ) -> torch.Tensor:
        if (
            x.shape[0] > self.TILED_ABOVE_FP8 and self._on_device(x)
            and (x.shape[0] > self.GROUPED_MAX_TOKENS or self._tiled_has(x.shape[0]))
        ):
            return self._sorted(x)
        out = self._grouped(x)
        if out is not None:
            return out
        T, H = x.shape
        router = F.linear(x.float(), self.gate.weight.float())  # [T, E]
        weights, selected = torch.topk(router, self.top_k, dim=-1)
        weights = torch.softmax(weights, dim=-1).to(x.dtype)  # [T, k]
        if T <= 256:
            # decode-sized batches: run EVERY expert densely. At these M
            # the expert GEMMs are weight-bound, and a batch this size
            # activates nearly all experts anyway — so the HBM cost is
            # the same as the sparse gather path, but there are no
            # dynamic shapes (topk/nonzero gathers), which is what lets
            # the decode step be hipGraph-captured. (The sparse path's
            # nonzero() aborts capture -> Mixtral decoded EAGER before
            # this: 47 ms/step of launch overhead.)
            wfull = torch.zeros(T, self.n_experts, dtype=x.dtype,
                                device=x.device)
            wfull.scatter_(1, selected, weights)
            fp8 = hasattr(self.experts[0].gate_up_proj, "forward_quantized")
            if fp8:
                xq, xs = ops.quant_fp8(x)
            out = None
            for e in range(self.n_experts):
                contrib = (
                    self.experts[e]((xq, xs)) if fp8 else self.experts[e](x)
                )
                contrib = contrib * wfull[:, e : e + 1]
                out = contrib if out is None else out + contrib
            return out
        # fp8 experts: quantize the hidden ONCE per layer and hand each
        # expert a row gather of the shared (fp8, scale) pair — per-expert
        # dynamic quantization costs more in launches than fp8 wins back
        # (measured: naive fp8 Mixtral 517 vs 769 bf16 tok/s, NOTES.md)
        fp8 = hasattr(self.experts[0].gate_up_proj, "forward_quantized")
        if fp8:
            xq, xs = ops.quant_fp8(x)
            xq_bytes = xq.view(torch.uint8)  # float8 lacks index_select
        out = torch.zeros_like(x)
        for e in range(self.n_experts):
            mask = selected == e  # [T, k]
            tok_idx, k_idx = mask.nonzero(as_tuple=True)
            if tok_idx.numel() == 0:
                continue
            if fp8:
                sub = (xq_bytes[tok_idx].view(xq.dtype), xs[tok_idx])
                contrib = self.experts[e](sub)
            else:
                contrib = self.experts[e](x[tok_idx])
            out.index_add_(0, tok_idx, contrib * weights[tok_idx, k_idx, None])
        return out


class DecoderLayer(nn.Module):
    def __init__(self, cfg: ModelArchConfig, layer_idx: int):
        super().__init__()
        self.input_layernorm = nn.Parameter(torch.ones(cfg.hidden_size))
        self.post_attention_layernorm = nn.Parameter(torch.ones(cfg.hidden_size))
        self.self_attn = Attention(cfg, layer_idx)
        self.mlp = (
            MoEMLP(cfg) if cfg.num_local_experts > 0 else MLP(cfg, layer_idx)
        )
        self.eps = cfg.rms_norm_eps
        # gemma2: branch outputs are normed BEFORE the residual add, with
        # separate pre/post feed-forward norms (4 norms per layer)
        self.post_norms = cfg.post_norms
        # granite: branch outputs scale by residual_multiplier before the
        # residual add
        self.res_mult = cfg.residual_multiplier or 1.0
        if cfg.post_norms:
            self.pre_feedforward_layernorm = nn.Parameter(
                torch.ones(cfg.hidden_size)
            )
            self.post_feedforward_layernorm = nn.Parameter(
                torch.ones(cfg.hidden_size)
            )

    def forward(self, x, residual, fb, kv_cache, cos_sin, as_sums: bool = False):
        """as_sums: the caller takes the branch as ops.ProductSums too, or with
        post norms as ops.BranchNorm (x may be that in any case)."""
        # products are handed on as sums in steps of few rows only
        branch = _branch if x.shape[0] <= ops.MAX_SUM_ROWS else _call
        last = branch if as_sums else _call
        if self.post_norms:
            # incoming invariant: hidden = x + residual (residual None at
            # layer 0); outgoing (m_normed, hidden_after_attn) keeps it,
            # so the model-level final fused_add_rmsnorm still applies
            if residual is None:
                hidden, x = x, ops.rmsnorm(x, self.input_layernorm, self.eps)
            else:
                x, hidden = ops.add_and_norm(x, residual, self.input_layernorm, self.eps)
            a = branch(self.self_attn, x, fb, kv_cache, cos_sin)
            x, h2 = ops.add_and_norm(
                ops.BranchNorm(a, self.post_attention_layernorm, self.eps), hidden,
                self.pre_feedforward_layernorm, self.eps,
            )
            mm = branch(self.mlp, x, fb)
            if as_sums:  # the next layer's (or the final) norm takes this one too
                return ops.BranchNorm(mm, self.post_feedforward_layernorm, self.eps), h2
            return ops.rmsnorm(mm, self.post_feedforward_layernorm, self.eps), h2
        if (
            getattr(self, "_fp8_fused", False)
            and x.is_cuda
            and fb.lora_ids is None
        ):
            # fp8 serving: norms/activations emit fp8 + per-row scales
            # directly (row_ops.hip), so activation quantization costs
            # nothing extra; residual stays bf16
            if residual is None:
                residual = x
                xq, xs = ops.rmsnorm_fp8(x, self.input_layernorm, self.eps)
            else:
                xq, xs = ops.fused_add_rmsnorm_fp8(
                    x, residual, self.input_layernorm, self.eps
                )
            x = branch(self.self_attn, (xq, xs), fb, kv_cache, cos_sin)
            if isinstance(self.mlp, MoEMLP):
                # router consumes bf16; MoEMLP quantizes once internally
                x, residual = ops.fused_add_rmsnorm(
                    x, residual, self.post_attention_layernorm, self.eps
                )
                x = self.mlp(x)
            else:
                xq, xs = ops.fused_add_rmsnorm_fp8(
                    x, residual, self.post_attention_layernorm, self.eps
                )
                x = last(self.mlp, (xq, xs), fb=fb)
            return x, residual
        if residual is None:
            residual = x
            x = ops.rmsnorm(x, self.input_layernorm, self.eps)
        else:
            x, residual = ops.fused_add_rmsnorm(
                x, residual, self.input_layernorm, self.eps
            )
        plain = self.res_mult == 1.0  # the next norm reads the branch as it is
        x = (branch if plain else _call)(self.self_attn, x, fb, kv_cache, cos_sin)
        if self.res_mult != 1.0:
            x = x * self.res_mult
        x, residual = ops.fused_add_rmsnorm(
            x, residual, self.post_attention_layernorm, self.eps
        )
        x = (last if plain else _call)(self.mlp, x, fb)
        if self.res_mult != 1.0:
            x = x * self.res_mult
        return x, residual


class LlamaForCausalLM(nn.Module):
    """Covers dense Llama and (with num_local_experts>0) Mixtral MoE."""

    def __init__(self, cfg: ModelArchConfig, device=None, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        # build weights directly in the target dtype/device: a 70B model
        # constructed fp32-first would transiently need ~280 GB
        prev_dtype = torch.get_default_dtype()
        torch.set_default_dtype(dtype)
        try:
            with torch.device(device if device is not None else "cpu"):
                self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
                self.layers = nn.ModuleList(
                    [DecoderLayer(cfg, i) for i in range(cfg.num_hidden_layers)]
                )
                self.norm = nn.Parameter(torch.ones(cfg.hidden_size))
                if cfg.tie_word_embeddings:
                    self.lm_head = None
                else:
                    self.lm_head = EngineLinear(
                        cfg.hidden_size, cfg.vocab_size, bias=False
                    )
        finally:
            torch.set_default_dtype(prev_dtype)
        from kubeai_amd.ops import ref as ops_ref

        self.register_buffer(
            "cos_sin",
            ops_ref.make_cos_sin_cache(
                cfg.head_dim, cfg.max_position_embeddings, cfg.rope_theta,
                rope_scaling=cfg.rope_scaling,
            ).to(device=device),
            persistent=False,
        )
        if cfg.rope_local_base_freq:
            # gemma3: windowed layers rope with the LOCAL base, unscaled
            self.register_buffer(
                "cos_sin_local",
                ops_ref.make_cos_sin_cache(
                    cfg.head_dim, cfg.max_position_embeddings,
                    cfg.rope_local_base_freq,
                ).to(device=device),
                persistent=False,
            )
        else:
            self.cos_sin_local = None

    @torch.inference_mode()
    def forward(self, fb: ForwardBatch) -> torch.Tensor:
        cs = (
            (self.cos_sin, self.cos_sin_local)
            if self.cos_sin_local is not None
            else self.cos_sin
        )
        x = self.embed_tokens(fb.input_ids.long())
        if self.cfg.scale_embeddings:
            # gemma: embeddings scaled by sqrt(hidden), cast to model dtype
            # first (HF normalizer semantics)
            x = x * torch.tensor(
                self.cfg.hidden_size ** 0.5, dtype=x.dtype
            )
        elif self.cfg.embedding_multiplier:
            x = x * self.cfg.embedding_multiplier  # granite
        if fb.mm_embeds is not None:
            # image-placeholder positions take the vision-tower embeddings
            x = x.index_copy(0, fb.mm_idx, fb.mm_embeds.to(x.dtype))
        fb.decode_plans = {}
        try:
            return self._run_layers(x, fb, cs)
        finally:
            fb.decode_plans = None

    def _run_layers(self, x, fb, cs):
        residual = None
        n = len(self.layers)
        # layers that nobody else looks at hand on products that the next one's
        # (or the final) norm adds up
        few = x.shape[0] <= ops.MAX_SUM_ROWS or self.cfg.post_norms
        own = [few and type(layer) is DecoderLayer and not _hooked(layer)
               for layer in self.layers]
        for i, layer in enumerate(self.layers):
            kw = {"as_sums": True} if own[i] and (i + 1 == n or own[i + 1]) else {}
            x, residual = layer(x, residual, fb, self.kv_caches[i], cs, **kw)
        if isinstance(x, ops.BranchNorm):  # (sums in fp32, as fused_add_rmsnorm's)
            x = ops.rmsnorm(x.x, x.weight, x.eps)
        x, _ = ops.fused_add_rmsnorm(x, residual, self.norm, self.cfg.rms_norm_eps)
        return x

    @torch.inference_mode()
    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        if self.lm_head is None:
            logits = F.linear(hidden, self.embed_tokens.weight).float()
        else:
            logits = self.lm_head(hidden).float()
        if self.cfg.logits_scaling:
            logits = logits / self.cfg.logits_scaling  # granite
        cap = self.cfg.final_logit_softcap
        if cap > 0:
            logits = cap * torch.tanh(logits / cap)
        return logits

    def bind_kv_caches(self, kv_caches: list[tuple[torch.Tensor, torch.Tensor]]):
        self.kv_caches = kv_caches
