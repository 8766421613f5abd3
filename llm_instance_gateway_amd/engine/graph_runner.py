"""hipGraph capture of decode-only steps.

MI355X-first use of HIP graphs instead of a tracing compiler (build brief):
a decode step of Llama-3-8B issues ~400 kernels (32 layers x {norm, rope,
cache-scatter, attention, 4 GEMMs, swiglu, 2x SGMV x 4 modules}); dispatched
eagerly from Python the GPU sits ~50-60% idle (profiles/r01_*.md).  Decode
batches have a fixed shape per batch-size bucket, so the whole step is
captured once per bucket into a hipGraph and replayed with one launch.

Static-buffer contract: per padded batch size B the graph reads
  ids[B], pos[B], slot_mapping[B], block_tables[B, MAXB], context_lens[B],
  lora_slots[B]
and writes logits[B, vocab] (bf16).  Padding rows decode a scratch KV block
(one extra block appended to the cache pool) with context_len=1 so they
compute garbage without touching live state.  The inputs of a bucket lie in
one device buffer, so a replay needs one copy from the host.

Prefill / mixed steps stay eager (their shapes vary too much to bucket).
"""

from __future__ import annotations

import gc
import logging
from types import SimpleNamespace
from typing import Dict, List, Optional

import numpy as np
import torch

from .batch_arrays import decode_lora_rows, decode_slots, device_view, lay_out, pack_decodes
from .metadata import BatchMeta

log = logging.getLogger(__name__)

CAPTURE_SIZES = [1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256, 320, 384, 448, 512]


class DecodeGraphRunner:
    def __init__(self, runner) -> None:
        self.runner = runner
        self.device = runner.device
        cfg = runner.config
        mc = cfg.model
        self.max_bs = cfg.max_num_seqs
        self.max_blocks = cfg.max_model_len // cfg.block_size
        self.block_size = cfg.block_size
        self.sizes = [s for s in CAPTURE_SIZES if s <= self.max_bs]
        if self.sizes[-1] != self.max_bs:
            self.sizes.append(self.max_bs)
        dev = self.device
        B = self.max_bs
        # graph-private LoRA shrink workspace (see metadata.lora_ws): replay
        # must not share u with a concurrently-running eager prefill
        self.lora_ws: Optional[torch.Tensor] = None
        # Models that address the batch per sequence (general-size attention,
        # recurrent layers): a decode step is B one-token segments, row i ==
        # sequence i; only the state slot and the starts-here flag vary.
        self.seq_tables = bool(getattr(runner.model, "needs_seq_tables", False))
        if self.seq_tables:
            ar = torch.arange(B, dtype=torch.int32, device=dev)
            self.tok_seq = ar.clone()
            self.seg_start = ar.clone()
            self.seg_len = torch.ones(B, dtype=torch.int32, device=dev)
            # scratch state slot for padding rows = one past the pool
            self.scratch_slot = getattr(runner, "num_state_slots", 0)
        # scratch KV block for padding rows = last block of the (extended) pool
        self.scratch_block = runner.config.num_kv_blocks  # extra block id
        self.graphs: Dict[int, torch.cuda.CUDAGraph] = {}
        self.logits: Dict[int, torch.Tensor] = {}
        self._pool = None
        self._inputs: Dict[int, SimpleNamespace] = {}
        self.with_lora = False
        self.lora_in_layer = False

    def _graph_nsplits(self, B: int) -> int:
        """How many parts a bucket's decode walks may be cut into: a replay's
        launches are fixed, so this follows from the bucket's size and the
        engine's longest context.  The kernel takes fewer where a row is short
        (at least 512 keys a part); the other workgroups leave at once."""
        from .. import ops

        shape = self._attn_shape()
        if shape is None:
            return 1
        return ops.decode_nsplits(B, shape[1], self.max_blocks * self.block_size)

    def _attn_shape(self):
        """(q heads, kv heads, head size) of the layers that run the split
        paged-decode kernel; None when no layer does."""
        model = self.runner.model
        if hasattr(model, "decode_attention_shape"):
            return model.decode_attention_shape()
        attn = model.layers[0].self_attn
        return attn.num_heads, attn.num_kv_heads, attn.head_dim

    def _fields(self, B: int) -> dict:
        """name -> (dtype, shape) of what a bucket's graph reads anew each replay."""
        f = dict(ids=(torch.int64, (B,)), pos=(torch.int64, (B,)), slot_mapping=(torch.int64, (B,)),
                 block_tables=(torch.int32, (B, self.max_blocks)), context_lens=(torch.int32, (B,)))
        if self.seq_tables:
            f.update(seg_slot=(torch.int32, (B,)), seg_fresh=(torch.int32, (B,)))
        if self.with_lora and self.lora_in_layer:
            # row tiles, as many as B tokens can need, the unused ones empty
            n = self._max_rows(B)
            f.update(lora_tok=(torch.int32, (n, 16)), lora_len=(torch.int32, (n,)), lora_slot=(torch.int32, (n,)))
        elif self.with_lora:
            # slot-grouped SGMV units, empty ones padded with length 0
            f.update(lora_slots=(torch.int32, (B,)), lora_order=(torch.int32, (B,)), lora_t0=(torch.int32, (B,)),
                     lora_len=(torch.int32, (B,)), lora_slot=(torch.int32, (B,)))
        return f

    def _views(self, B: int) -> SimpleNamespace:
        """A bucket's inputs: `dev` tensors, the `host` arrays they are copied
        from, and the two byte ranges that the copy moves."""
        if B not in self._inputs:
            fields = self._fields(B)
            offsets, total = lay_out(fields.values())
            dev, host = SimpleNamespace(), SimpleNamespace()
            for (name, (dtype, shape)), o in zip(fields.items(), offsets):
                setattr(dev, name, device_view(self._dev, o, dtype, shape))
                setattr(host, name, device_view(self._host, o, dtype, shape).numpy())
            self._inputs[B] = SimpleNamespace(dev=dev, host=host, to=self._dev[:total], src=self._host[:total])
        return self._inputs[B]

    def _meta(self, B: int) -> BatchMeta:
        x = self._views(B).dev
        extra = {}
        if self.seq_tables:
            extra = dict(
                seq_block_tables=x.block_tables,
                tok_seq=self.tok_seq[:B],
                seg_start=self.seg_start[:B],
                seg_len=self.seg_len[:B],
                seg_slot=x.seg_slot,
                seg_fresh=x.seg_fresh,
                seg_ctx=x.context_lens,
                max_seg_len=1,
            )
        if self.with_lora and self.lora_in_layer:
            extra.update(lora_rows_tok=x.lora_tok, lora_rows_len=x.lora_len, lora_rows_slot=x.lora_slot)
        elif self.with_lora:
            extra.update(
                lora_slot_per_token=x.lora_slots,
                lora_order=x.lora_order,
                lora_unit_t0=x.lora_t0,
                lora_unit_len=x.lora_len,
                lora_unit_slot=x.lora_slot,
            )
        return BatchMeta(
            **extra,
            num_prefill_tokens=0,
            num_decode_tokens=B,
            slot_mapping=x.slot_mapping,
            decode_block_tables=x.block_tables,
            decode_context_lens=x.context_lens,
            lora_ws=self.lora_ws,
            decode_nsplits=self._graph_nsplits(B),
        )

    def _max_rows(self, B: int) -> int:
        from ..lora.manager import max_lora_rows

        return max_lora_rows(B, self.runner.adapter_manager.max_slots)

    def _plain_head(self) -> bool:
        """Whether compute_logits is nothing but head_logits of the rows asked
        for, in fp32: not where it was overridden without the other."""
        model = self.runner.model
        for owner in (model, *type(model).__mro__):
            if "compute_logits" in vars(owner):
                return "head_logits" in vars(owner)
        return False

    def _forward(self, B: int) -> torch.Tensor:
        model = self.runner.model
        x = self._views(B).dev
        hidden = model(x.ids, x.pos, self.runner.kv_caches, self._meta(B))
        if self._plain_head():
            return model.head_logits(hidden).to(self.runner.dtype)
        idx = torch.arange(B, device=self.device)
        return model.compute_logits(hidden, idx).to(self.runner.dtype)

    def capture(self, with_lora: bool) -> None:
        self.with_lora = with_lora
        mgr = self.runner.adapter_manager
        # (not over modules whose hooks or replaced forwards belong into the graph)
        self.lora_in_layer = with_lora and getattr(mgr, "in_layer", False) and self.runner.model.plain_layers()
        # one buffer for the inputs of any bucket (the largest needs the most)
        total = lay_out(self._fields(self.max_bs).values())[1]
        self._dev = torch.zeros(total, dtype=torch.uint8, device=self.device)
        self._host = torch.zeros(total, dtype=torch.uint8, pin_memory=True)
        self._inputs = {}
        if with_lora and self.lora_ws is None:
            self.lora_ws = torch.zeros(
                self.max_bs, mgr.rank, dtype=mgr.dtype, device=self.device
            )
        # Preallocate the flash-decode split scratch at the max any bucket
        # needs so every captured graph bakes one stable pointer (the ops
        # cache grows monotonically; growth during capture would leave
        # earlier graphs pointing at freed memory).
        from .. import ops

        shape = self._attn_shape()
        hq, d = (shape[0], shape[2]) if shape is not None else (0, 0)
        max_scratch = max(
            (B * hq * self._graph_nsplits(B) * (d + 2) for B in self.sizes),
            default=0,
        )
        if max_scratch > 0 and self.device.type == "cuda":
            ops.split_scratch(self.device, max_scratch)
        torch.cuda.synchronize(self.device)
        # Warmup on a side stream (torch.cuda.graph requirement) — at EVERY
        # capture batch size: hipBLASLt picks its algorithm + allocates its
        # workspace on the FIRST call of each GEMM shape, and a first call
        # that happens inside graph capture is restricted to slow no-workspace
        # fallbacks which then get baked into the graph (measured: in-graph
        # decode GEMMs 2-8x slower than the same shapes eager —
        # profiles/r01_c256_breakdown.md).
        s = torch.cuda.Stream(device=self.device)
        s.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(s):
            for B in self.sizes:
                self._fill(B, [], None)  # padding rows only
                self._forward(B)
                s.synchronize()  # before the next bucket's rows overwrite the host's
        torch.cuda.current_stream(self.device).wait_stream(s)
        torch.cuda.synchronize(self.device)
        # Graphs of an engine that is no longer referenced sit in reference
        # cycles; if the collector freed one of them in the middle of a
        # capture, its destructor would call into the runtime, which is not
        # permitted then and ends the process.  Collect now, and hold the
        # collector off until the captures are done.
        gc.collect()
        gc_was_on = gc.isenabled()
        gc.disable()
        try:
            for B in self.sizes:
                g = torch.cuda.CUDAGraph()
                if self._pool is None:
                    with torch.cuda.graph(g):
                        self.logits[B] = self._forward(B)
                    self._pool = g.pool()
                else:
                    with torch.cuda.graph(g, pool=self._pool):
                        self.logits[B] = self._forward(B)
                self.graphs[B] = g
        finally:
            if gc_was_on:
                gc.enable()
        torch.cuda.synchronize(self.device)
        log.info("captured %d decode graphs (lora=%s)", len(self.graphs), with_lora)

    def pick_size(self, n: int) -> Optional[int]:
        for s in self.sizes:
            if s >= n:
                return s
        return None

    def run(
        self,
        decodes,  # List[ScheduledSeq]
        slot_of,  # callable(name) -> int, or None
    ) -> torch.Tensor:
        """Fill the bucket's inputs, replay its graph, return logits[:n]."""
        n = len(decodes)
        B = self.pick_size(n)
        assert B is not None
        self._fill(B, decodes, slot_of)
        self.graphs[B].replay()
        return self.logits[B][:n]

    def _fill(self, B: int, decodes, slot_of) -> None:
        """The inputs of `decodes`, padding rows behind them, to the device."""
        n, bs = len(decodes), self.block_size
        v = self._views(B)
        x = v.host
        seqs = [ss.seq for ss in decodes]
        x.ids[n:] = 0
        x.pos[n:] = 0
        x.block_tables[:] = 0  # another bucket's arrays lay here
        pack_decodes(seqs, bs, x.ids[:n], x.pos[:n], x.block_tables[:n])
        x.block_tables[n:, 0] = self.scratch_block
        decode_slots(x.pos, x.block_tables, bs, x.slot_mapping, x.context_lens)
        if self.seq_tables:
            x.seg_slot[:n] = [max(q.state_slot, 0) for q in seqs]
            x.seg_slot[n:] = self.scratch_slot
            x.seg_fresh[:] = x.pos == 0
        if self.with_lora and self.lora_in_layer:
            decode_lora_rows(seqs, slot_of, B, x.lora_tok, x.lora_len, x.lora_slot)
        elif self.with_lora:
            from ..lora.manager import build_lora_units

            slots = np.full(B, -1, dtype=np.int32)
            of = {name: slot_of(name) if name else -1 for name in {q.lora_name for q in seqs}}
            slots[:n] = [of[q.lora_name] for q in seqs]
            x.lora_slots[:] = slots
            x.lora_order[:], ut0, ulen, uslot = build_lora_units(slots)
            u = len(ut0)
            x.lora_t0[:u] = ut0
            x.lora_t0[u:] = 0
            x.lora_len[:u] = ulen
            x.lora_len[u:] = 0  # padding units: no-op in the kernels
            x.lora_slot[:u] = uslot
            x.lora_slot[u:] = -1
        v.to.copy_(v.src, non_blocking=True)
