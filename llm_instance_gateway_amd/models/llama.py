"""Llama-family dense transformer with paged-KV attention.

The model family the reference's fleet configs pin
(`examples/poc/manifests/vllm/vllm-lora-deployment.yaml`: Llama-2-7b;
Llama-3-8B / 70B).  Built MI355X-first:

  * flat unpadded token batches (prefill chunks + decodes in one forward);
  * custom CDNA4 kernels via the ops layer for RMSNorm (fused residual add),
    RoPE, KV-cache scatter, paged prefill/decode attention and SwiGLU;
  * the projections by `ops.linear`: a kernel of this package up to 1024 rows, of
    long weights 1792, where it is the faster one, library GEMMs elsewhere; LoRA deltas ride the SGMV path (`..lora`);
  * optional tensor parallelism: column-sharded QKV/gate-up, row-sharded
    O/down with one RCCL all-reduce per block over xGMI (`..parallel`).

Weights are random-init (no network — synthetic serving benchmark).
"""

from __future__ import annotations

import math
from typing import List

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from .. import ops
from ..engine.metadata import BatchMeta
from .config import ModelConfig


def _plain(d: dict) -> bool:
    """Whether calling the module with these attributes runs its class's forward
    and nothing else, so that kernels may take its place."""
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d)


def _linear(in_f: int, out_f: int, device, dtype) -> nn.Linear:
    lin = nn.Linear(in_f, out_f, bias=False, device="meta", dtype=dtype)
    lin = lin.to_empty(device=device)
    # cheap bounded init (never materialize fp32 copies of 8B params)
    with torch.no_grad():
        lin.weight.uniform_(-0.02, 0.02)
    return lin


def _product_alone(m: nn.Module) -> bool:
    """Whether m(x) is x @ m.weight.T and nothing else, its weight a parameter."""
    p = m._parameters
    return (type(m) is nn.Linear and _plain(m.__dict__) and p.get("weight") is not None and p.get("bias", p) is None
            and not _has_any_global_hook())


def _project(m: nn.Module, x: torch.Tensor, product=ops.linear) -> torch.Tensor:
    """m(x); a plain linear layer's product by `ops.linear` (or `ops.linear_parts`)."""
    return product(x, m._parameters["weight"]) if _product_alone(m) else m(x)


def _served(m: nn.Module, rows: int) -> bool:
    """Whether `_project` of that many rows runs on our kernels, in parts."""
    return _product_alone(m) and ops.linear_served(rows, m._parameters["weight"])


class Attention(nn.Module):
    def __init__(self, cfg: ModelConfig, device, dtype, tp=None) -> None:
        super().__init__()
        self.cfg = cfg
        self.tp = tp
        tp_size = tp.world_size if tp is not None else 1
        assert cfg.num_heads % tp_size == 0 and cfg.num_kv_heads % tp_size == 0
        self.num_heads = cfg.num_heads // tp_size
        self.num_kv_heads = cfg.num_kv_heads // tp_size
        self.head_dim = cfg.head_dim
        self.scale = 1.0 / math.sqrt(cfg.head_dim)
        h = cfg.hidden_size
        q_out = self.num_heads * self.head_dim
        kv_out = self.num_kv_heads * self.head_dim
        self.qkv_proj = _linear(h, q_out + 2 * kv_out, device, dtype)
        self.o_proj = _linear(q_out, h, device, dtype)
        self.q_size = q_out
        self.kv_size = kv_out
        # multi-LoRA hook (set by lora.manager.AdapterManager._attach)
        self._lora = None
        self._layer_idx = -1

    def forward(
        self,
        hidden: torch.Tensor,  # [T, H]
        positions: torch.Tensor,  # [T]
        kv_cache,  # (k_cache, v_cache) for this layer
        meta: BatchMeta,
        cos_sin_cache: torch.Tensor,
    ) -> torch.Tensor:
        qkv = _project(self.qkv_proj, hidden)
        if self._lora is not None:
            self._lora.apply(self._layer_idx, "qkv", hidden, qkv, meta)
        k_cache, v_cache = kv_cache
        q = ops.qkv_rope_cache(
            qkv, positions, cos_sin_cache, k_cache, v_cache, meta.slot_mapping, self.num_heads
        )
        attn_flat = self.attend(q, kv_cache, meta)
        o = _project(self.o_proj, attn_flat)
        if self._lora is not None:
            self._lora.apply(self._layer_idx, "o", attn_flat, o, meta)
        if self.tp is not None:
            o = self.tp.all_reduce(o)
        return o

    def attend(self, q: torch.Tensor, kv_cache, meta: BatchMeta) -> torch.Tensor:
        """Attention of the rotated queries [T, heads * D] over the paged cache."""
        k_cache, v_cache = kv_cache
        qh = q.view(-1, self.num_heads, self.head_dim)
        np_, nd = meta.num_prefill_tokens, meta.num_decode_tokens
        out = torch.empty_like(qh)
        if np_ > 0:
            ops.paged_attention_prefill(
                qh[:np_],
                k_cache,
                v_cache,
                meta.prefill_block_tables,
                meta.prefill_query_start_locs,
                meta.prefill_context_lens,
                self.scale,
                tok_block_tables=meta.prefill_tok_block_tables,
                tok_context_lens=meta.prefill_tok_context_lens,
                tile_seq=meta.prefill_tile_seq,
                tile_qstart=meta.prefill_tile_qstart,
                out=out[:np_],
            )
        if nd > 0:
            # slice end is explicit: the flat batch may carry GEMM-bucketing
            # pad rows after the decode partition
            ops.paged_attention_decode(
                qh[np_:np_ + nd],
                k_cache,
                v_cache,
                meta.decode_block_tables,
                meta.decode_context_lens,
                self.scale,
                max_ctx=meta.max_decode_ctx,
                nsplits=meta.decode_nsplits,
                out=out[np_:np_ + nd],
            )
        return out.view(-1, self.num_heads * self.head_dim)


class MLP(nn.Module):
    def __init__(self, cfg: ModelConfig, device, dtype, tp=None) -> None:
        super().__init__()
        self.tp = tp
        tp_size = tp.world_size if tp is not None else 1
        assert cfg.intermediate_size % tp_size == 0
        inter = cfg.intermediate_size // tp_size
        h = cfg.hidden_size
        # gate and up fused into one GEMM (silu_and_mul splits them)
        self.gate_up_proj = _linear(h, 2 * inter, device, dtype)
        self.down_proj = _linear(inter, h, device, dtype)
        self._lora = None
        self._layer_idx = -1

    def forward(self, x: torch.Tensor, meta=None) -> torch.Tensor:
        gu = _project(self.gate_up_proj, x)
        if self._lora is not None:
            self._lora.apply(self._layer_idx, "gate_up", x, gu, meta)
        act = ops.silu_and_mul(gu)
        y = _project(self.down_proj, act)
        if self._lora is not None:
            self._lora.apply(self._layer_idx, "down", act, y, meta)
        if self.tp is not None:
            y = self.tp.all_reduce(y)
        return y


class DecoderLayer(nn.Module):
    def __init__(self, cfg: ModelConfig, device, dtype, tp=None) -> None:
        super().__init__()
        self.input_layernorm = nn.Parameter(torch.ones(cfg.hidden_size, device=device, dtype=dtype))
        self.post_attention_layernorm = nn.Parameter(
            torch.ones(cfg.hidden_size, device=device, dtype=dtype)
        )
        self.eps = cfg.rms_norm_eps
        self.self_attn = Attention(cfg, device, dtype, tp)
        self.mlp = MLP(cfg, device, dtype, tp)

    def forward(self, hidden, residual, positions, kv_cache, meta, cos_sin_cache):
        if residual is None:
            residual = hidden
            h = ops.rms_norm(hidden, self.input_layernorm, self.eps)
        else:
            h, residual = ops.fused_add_rms_norm(
                hidden, residual, self.input_layernorm, self.eps
            )
        h = self.self_attn(h, positions, kv_cache, meta, cos_sin_cache)
        h, residual = ops.fused_add_rms_norm(
            h, residual, self.post_attention_layernorm, self.eps
        )
        h = self.mlp(h, meta)
        return h, residual


class LlamaForCausalLM(nn.Module):
    def __init__(self, cfg: ModelConfig, device="cpu", dtype=torch.bfloat16, tp=None) -> None:
        super().__init__()
        self.cfg = cfg
        self.tp = tp
        self.device_ = torch.device(device)
        self.dtype_ = dtype
        self.embed_tokens = nn.Embedding(
            cfg.vocab_size, cfg.hidden_size, device="meta", dtype=dtype
        ).to_empty(device=device)
        with torch.no_grad():
            self.embed_tokens.weight.uniform_(-0.02, 0.02)
        self.layers = nn.ModuleList(
            [DecoderLayer(cfg, device, dtype, tp) for _ in range(cfg.num_layers)]
        )
        self.norm = nn.Parameter(torch.ones(cfg.hidden_size, device=device, dtype=dtype))
        if cfg.tie_word_embeddings:
            self.lm_head = None
        else:
            self.lm_head = _linear(cfg.hidden_size, cfg.vocab_size, device, dtype)
        self.cos_sin_cache = ops.build_cos_sin_cache(
            cfg.head_dim, cfg.max_position_embeddings, cfg.rope_theta, device
        ).to(dtype=torch.float32)

    def forward(
        self,
        input_ids: torch.Tensor,  # [T]
        positions: torch.Tensor,  # [T]
        kv_caches: List,  # per layer (k_cache, v_cache)
        meta: BatchMeta,
    ) -> torch.Tensor:
        hidden = self.embed_tokens(input_ids)
        # (a graph being captured brings row tiles only where plain_layers() allowed them)
        if meta.lora_rows_tok is not None and (meta.lora_slot_per_token is None or self.plain_layers()):
            return self._forward_lora(hidden, positions, kv_caches, meta)
        if hidden.shape[0] == 1 and meta.lora_slot_per_token is None and self._row_products():
            return self._forward_row(hidden, positions, kv_caches, meta)
        if meta.lora_slot_per_token is None and self._open_norms(len(hidden)):
            return self._forward_open(hidden, positions, kv_caches, meta)
        residual = None
        for layer, kv in zip(self.layers, kv_caches):
            hidden, residual = layer(
                hidden, residual, positions, kv, meta, self.cos_sin_cache
            )
        hidden, _ = ops.fused_add_rms_norm(hidden, residual, self.norm, self.cfg.rms_norm_eps)
        return hidden

    def plain_layers(self) -> bool:
        """Whether the layers, their attention and feed-forward modules run this
        file's forwards and nothing else: no forward hook, no other class, no
        forward of an instance's own that kernels in their place would pass by.
        Asked on every eager step, so it goes by the modules' dictionaries."""
        if _has_any_global_hook():
            return False
        for layer in self.layers:
            if type(layer) is not DecoderLayer or not _plain(layer.__dict__):
                return False
            parts = layer.__dict__["_modules"]
            attn, mlp = parts["self_attn"], parts["mlp"]
            if type(attn) is not Attention or type(mlp) is not MLP:
                return False
            if not (_plain(attn.__dict__) and _plain(mlp.__dict__)):
                return False
        return True

    def batch_rows(self, tokens: int, multiple: int, lora_tiles: int | None = None) -> int:
        """Rows to pad a flat batch of tokens to; `lora_tiles`: of a step with adapters,
        its tiles of rows, 0 where adapters have kernels of their own.

        The library's products want few, tile-friendly counts, those of `ops.linear`
        take any: none is added where all of a layer's projections run there (786
        tokens: a step of 8B widths takes 4.6 ms, 5.1 padded to 832 with qkv and gate_up
        at the library), few where some do.  At such a count those left to the library
        miss its tuned table, which knows multiples of 256: the rows saved are worth
        more.  Under 2^20 weights a projection takes its launch's time at either count,
        and the multiple stays.

        Where norms and rotation do not add up parts (sharded layers, hooks, adapters of
        their own kernels or of many tiles) every product has to come rounded, for which
        fewer run here: at 786 rows of 8B widths qkv and o are the library's.  By itself a
        step takes the same time at any such count (786 rows of adapters of rank 32 4881
        us, 832 4933; 1000 5418, 1024 5389), but each count that the library meets for the
        first time costs it 70 us a product: 12 multiples of 64 against 768 counts.

        From 1025 to 2048 rows a step is mostly the library's products, and of its untuned
        counts not every multiple of 64 is a good one: 1600 rows of 8B widths 6956 us, 1792
        6167.  Those of 128 are, all four of them measured at seven shapes of 2560 to 8192 columns
        (8B: 1152 rows 4591 us, 1280 4789; 1408 5137, 1536 5259; 1664 6064, 1792 6167; 1920
        6560, 2048 6620; 5 adapters: 1152 5015, 1280 5129).  At 2048 columns 1152 rows
        take up to 1.5 % longer than 1280, and the multiple stays, as for sharded layers,
        which were not measured."""
        if tokens > 1024:
            step = min(128, multiple) if tokens <= 2048 and self.tp is None and self.cfg.hidden_size > 2048 else multiple
            return -(-tokens // step) * step
        attn, mlp = self.layers[0].self_attn, getattr(self.layers[0], "mlp", None)
        modules = [attn.qkv_proj, attn.o_proj, *((mlp.gate_up_proj, mlp.down_proj) if type(mlp) is MLP else ())]
        served = [_served(m, tokens) and m.weight.numel() >= 1 << 20 for m in modules]
        here = [s and ops.linear_pays(tokens, m.weight) for s, m in zip(served, modules)]
        if here != served and self._in_parts(tokens, lora_tiles):
            here = served
        if all(here):
            return tokens
        step = min(64, multiple) if any(here) else multiple
        return -(-tokens // step) * step

    def _in_parts(self, tokens: int, lora_tiles: int | None) -> bool:
        """Whether what reads the products of such a step (`batch_rows`) adds up parts."""
        if lora_tiles is None:
            return self._open_norms(tokens)
        return (self.tp is None and lora_tiles > 0 and ops.lora_norm_opens(ops.BASE_ROWS, 16 * lora_tiles, self.cfg.hidden_size)
                and self.plain_layers())

    def _row_products(self) -> bool:
        """Whether every projection of a layer is one that `ops.row_product` serves."""
        if self.tp is not None or not self.plain_layers():
            return False
        most = ops.row_product_most(self.norm)
        for layer in self.layers:
            attn, mlp = layer.self_attn, layer.mlp
            for m, norm in ((attn.qkv_proj, True), (attn.o_proj, False), (mlp.gate_up_proj, True), (mlp.down_proj, False)):
                if type(m) is not nn.Linear or not _plain(m.__dict__):
                    return False
                p = m._parameters
                if p["bias"] is not None or not ops.row_product_serves(p["weight"], norm, most):
                    return False
        return True

    def _forward_row(self, hidden, positions, kv_caches, meta: BatchMeta) -> torch.Tensor:
        """The layers for a single token: norms, the activation, the rotation and what
        merges the parts of the attention's walk live in the projections' kernels."""
        residual, x = None, hidden
        rotates = self.cfg.head_dim % 64 == 0
        for layer, kv in zip(self.layers, kv_caches):
            attn, mlp = layer.self_attn, layer.mlp
            if rotates:
                q = ops.row_product_heads(
                    x, attn.qkv_proj.weight, layer.input_layernorm, layer.eps, residual, positions, self.cos_sin_cache, kv[0],
                    kv[1], meta.slot_mapping, attn.num_heads)
                q, residual = (q, x) if residual is None else q
            else:
                qkv = ops.row_product(x, attn.qkv_proj.weight, layer.input_layernorm, layer.eps, residual)
                qkv, residual = (qkv, x) if residual is None else qkv
                q = ops.qkv_rope_cache(
                    qkv, positions, self.cos_sin_cache, kv[0], kv[1], meta.slot_mapping, attn.num_heads)
            if meta.num_decode_tokens == 1 and "attend" not in attn.__dict__:
                a, parts = ops.paged_attention_decode_open(
                    q.view(1, attn.num_heads, -1), kv[0], kv[1], meta.decode_block_tables, meta.decode_context_lens, attn.scale,
                    meta.max_decode_ctx, meta.decode_nsplits)
            else:
                a, parts = attn.attend(q, kv, meta), None
            o = ops.row_product(a, attn.o_proj.weight, parts=parts)
            act, residual = ops.row_product(
                o, mlp.gate_up_proj.weight, layer.post_attention_layernorm, layer.eps, residual, silu=True)
            x = ops.row_product(act, mlp.down_proj.weight)
        hidden, _ = ops.fused_add_rms_norm(x, residual, self.norm, self.cfg.rms_norm_eps)
        return hidden

    def _open_norms(self, rows: int) -> bool:
        """Whether `_forward_open` is for a step of that many rows without adapters."""
        c = self.cfg
        return (self.tp is None and self.norm.is_cuda and self.norm.dtype == torch.bfloat16 and c.head_dim % 64 == 0
                and ops.lora_norm_opens(ops.BASE_ROWS, rows, c.hidden_size) and self.plain_layers()
                and self._open_weights(self.layers[0], rows) is not None)

    @staticmethod
    def _open_weights(layer: DecoderLayer, rows: int):
        """The weights of qkv, o, gate_up and down of a layer whose norms may leave
        their factor to what reads the products behind them, and come after products
        in parts: where all four are products and nothing else, by our kernels."""
        m = layer.__dict__["_modules"]
        attn, mlp = m["self_attn"].__dict__["_modules"], m["mlp"].__dict__["_modules"]
        out = []
        for lin in (attn["qkv_proj"], attn["o_proj"], mlp["gate_up_proj"], mlp["down_proj"]):
            if not _served(lin, rows):
                return None
            out.append(lin._parameters["weight"])
        return out if out[2].shape[0] % 64 == 0 else None

    def _forward_open(self, hidden, positions, kv_caches, meta: BatchMeta) -> torch.Tensor:
        """The layers with each norm as one kernel that adds up the product before
        it and leaves its factor to the rotation and the activation; layers that
        do more than multiply run their own forward."""
        rows = ops.BASE_ROWS
        layers = list(zip(self.layers, kv_caches))
        residual, y, weights = None, hidden, self._open_weights(layers[0][0], len(hidden))
        for i, (layer, kv) in enumerate(layers):
            after = self._open_weights(layers[i + 1][0], len(hidden)) if i + 1 < len(layers) else None
            if weights is None:
                y, residual = layer(y, residual, positions, kv, meta, self.cos_sin_cache)
                weights = after
                continue
            qkv, o, gate_up, down = weights
            h, _, norm = ops.lora_norm_open(y, residual, layer.input_layernorm, layer.eps, rows)
            if residual is None:
                residual = hidden
            attn = layer.self_attn
            q = ops.lora_qkv_rope_cache(
                ops.projection_parts(h, qkv), positions, self.cos_sin_cache, kv[0], kv[1], meta.slot_mapping,
                attn.num_heads, rows, None, None, norm)
            h, _, norm = ops.lora_norm_open(
                ops.projection_parts(attn.attend(q, kv, meta), o), residual, layer.post_attention_layernorm, layer.eps,
                rows)
            act = ops.lora_silu_and_mul(ops.linear(h, gate_up), rows, None, None, None, None, norm)
            y = (ops.linear if after is None else ops.projection_parts)(act, down)
            weights = after
        return ops.fused_add_rms_norm(y, residual, self.norm, self.cfg.rms_norm_eps)[0]

    def lora_in_layer(self, rank: int, dims: dict) -> bool:
        """Whether `_forward_lora` serves adapters of that rank over those
        modules: what the kernels of ops/csrc/lora_rows.hip take."""
        c = self.cfg
        return (
            rank == 16
            and set(dims) == {"qkv", "o", "gate_up", "down"}
            and c.hidden_size in ops.LORA_ROWS_WIDTHS
            and c.intermediate_size % 32 == 0
            and c.head_dim % 64 == 0
            and (c.num_heads * c.head_dim) % 32 == 0
        )

    def _forward_lora(self, hidden, positions, kv_caches, meta: BatchMeta) -> torch.Tensor:
        """The layers with every adapter's products carried by the kernels
        between the projections instead of kernels of their own: B u is added
        where a projection's output is read, A x formed where its input is
        written."""
        lora = self.layers[0].self_attn._lora
        rows = (meta.lora_rows_tok, meta.lora_rows_len, meta.lora_rows_slot)
        c = self.cfg
        ws, u_o, u_down = ops.lora_workspace(
            rows, c.hidden_size, c.num_heads * c.head_dim, c.intermediate_size)
        a, b = lora.a_stacks, lora.b_stacks
        residual, y, last = None, hidden, None
        # Norms whose readers can take the rows' factor themselves are one launch, and
        # add up the product before them.  Only products carry the factor through: a
        # module with a bias or a hook gets normed rows.  The rotation takes it with
        # fp32 parts only: a rounded product would be rounded once more on its way to V.
        can_open = ops.lora_norm_opens(rows, len(hidden), c.hidden_size)

        def open_in(i):  # the norm at layer i's entry
            return can_open and i < len(self.layers) and _served(self.layers[i].self_attn.qkv_proj, len(hidden))

        parts = open_in(0)
        for i, (layer, kv) in enumerate(zip(self.layers, kv_caches)):
            attn, mlp = layer.self_attn, layer.mlp
            opens = can_open and _product_alone(mlp.gate_up_proj)  # the norm behind the attention
            norm = ops.lora_norm_open if parts else ops.lora_rms_norm
            if last is None:
                h, u, *scale = norm(y, None, layer.input_layernorm, layer.eps, rows, a_stack=a[(i, "qkv")], u_out=ws)
                residual = hidden
            else:
                h, u, *scale = norm(
                    y, residual, layer.input_layernorm, layer.eps, rows, u_down, b[(last, "down")], a[(i, "qkv")], ws)
            q = ops.lora_qkv_rope_cache(
                _project(attn.qkv_proj, h, ops.linear_parts if parts else ops.linear), positions, self.cos_sin_cache,
                kv[0], kv[1], meta.slot_mapping, attn.num_heads, rows, u, b[(i, "qkv")], *scale)
            o = attn.attend(q, kv, meta)
            ops.lora_shrink(o, rows, a[(i, "o")], u_o)
            norm = ops.lora_norm_open if opens else ops.lora_rms_norm
            h, u, *scale = norm(
                _project(attn.o_proj, o, ops.linear_parts if opens else ops.linear), residual,
                layer.post_attention_layernorm, layer.eps, rows, u_o, b[(i, "o")], a[(i, "gate_up")], ws)
            act = ops.lora_silu_and_mul(
                _project(mlp.gate_up_proj, h), rows, u, b[(i, "gate_up")], a[(i, "down")], u_down, *scale)
            parts = open_in(i + 1)
            y, last = _project(mlp.down_proj, act, ops.linear_parts if parts else ops.linear), i
        return ops.lora_rms_norm(
            y, residual, self.norm, self.cfg.rms_norm_eps, rows, u_down, b[(last, "down")])[0]

    def head_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        """Logits of all rows, as the product leaves them."""
        w = self.embed_tokens.weight if self.lm_head is None else self.lm_head.weight
        # hidden is replicated across the TP group (each block ends in an
        # all-reduce), so every rank computes identical full-vocab logits.
        return ops.linear(hidden, w)

    def compute_logits(self, hidden: torch.Tensor, indices: torch.Tensor) -> torch.Tensor:
        """fp32 logits only at the sampled positions (last token of each
        finished chunk / each decode)."""
        return self.head_logits(hidden[indices]).float()
