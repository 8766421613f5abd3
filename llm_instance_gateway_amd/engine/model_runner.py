"""Model runner: owns the model, the physical paged KV cache, and one-step
execution (batch build → forward → sample).

MI355X notes: the KV cache is sized against the 288 GB HBM3E pool at engine
init (`determine_num_kv_blocks`); batches are flat/unpadded; all per-step
index tensors are built on host and copied in one piece.
"""

from __future__ import annotations

import logging
from typing import Dict, List, Optional, Tuple

import numpy as np
import torch

from ..models.config import ModelConfig
from ..utils.tunableop import eager_tuned
from .batch_arrays import pack_decodes, pack_rows, table_rows, upload
from .config import EngineConfig
from .metadata import BatchMeta
from ..utils.tracing import gpu_range
from .sampling import sample_tokens
from .scheduler import ScheduledSeq, SchedulerOutput
from .sequence import Sequence

log = logging.getLogger(__name__)


def build_model(cfg: ModelConfig, device, dtype, tp=None):
    """Instantiate the class registered for cfg.architecture (and load its
    checkpoint when the config names a folder)."""
    from ..models.registry import build_model as _build

    return _build(cfg, device, dtype, tp)


def determine_num_kv_blocks(
    config: EngineConfig, device: torch.device, tp_size: int = 1, elem_size: int = 2
) -> int:
    """Size the paged KV pool from free HBM after weights, honoring
    gpu_memory_utilization (the reference fleet runs vLLM at 0.95 —
    tools/dynamic-lora-sidecar/deployment.yaml:40)."""
    mc = config.model
    # K+V of every layer that keeps a paged cache (recurrent layers keep a
    # fixed-size state per slot instead, allocated separately)
    bytes_per_block = max(1, mc.kv_elems_per_token(tp_size) * config.block_size * elem_size)
    if device.type == "cuda":
        free, total = torch.cuda.mem_get_info(device)
        budget = int(total * config.gpu_memory_utilization) - (total - free)
        budget = max(budget, 0)
        n = budget // bytes_per_block
        return int(n)
    return config.num_kv_blocks


class ModelRunner:
    def __init__(
        self,
        config: EngineConfig,
        device: str = "cpu",
        dtype: torch.dtype = torch.bfloat16,
        tp=None,
    ) -> None:
        self.config = config
        self.device = torch.device(device)
        self.dtype = dtype
        self.tp = tp
        mc = config.model
        log.info("building model %s on %s", mc.name, self.device)
        self.model = build_model(mc, self.device, dtype, tp)
        if config.quant == "fp8":
            if mc.is_moe:
                raise ValueError("quant='fp8' covers dense models only")
            from ..models.quant import convert_linears_to_fp8

            n_q = convert_linears_to_fp8(self.model)
            if self.device.type == "cuda":
                torch.cuda.empty_cache()  # bf16 projection weights are gone
            log.info("fp8 quantization: %d projection GEMMs converted", n_q)
        tp_size = tp.world_size if tp is not None else 1
        if self.device.type == "cuda":
            n = determine_num_kv_blocks(
                config, self.device, tp_size, torch.empty((), dtype=dtype).element_size()
            )
            if n <= 0:
                raise RuntimeError("no HBM left for KV cache after weights")
            config.num_kv_blocks = min(
                n, config.num_kv_blocks if config.num_kv_blocks > 0 else n
            )
        kvh = mc.num_kv_heads // tp_size
        # +1 scratch block: hipGraph decode padding rows write their K/V there
        nblk = config.num_kv_blocks + 1
        self.num_state_slots = 0
        if hasattr(self.model, "cache_specs"):
            # Heterogeneous stack: every layer declares what it keeps — paged
            # K/V (key and value head sizes may differ) or an fp32 state
            # vector per slot (+1 scratch slot for padding rows).
            if mc.has_recurrent_state:
                self.num_state_slots = config.num_state_slots or config.max_num_seqs
            self.kv_caches = []

            def make(spec) -> tuple:
                if spec["kind"] == "kv":
                    g = spec["kv_heads"]
                    return (
                        torch.zeros((nblk, g, config.block_size, spec["k_dim"]), dtype=dtype, device=self.device),
                        torch.zeros((nblk, g, config.block_size, spec["v_dim"]), dtype=dtype, device=self.device),
                    )
                if spec["kind"] == "latent":
                    # one shared row per token: keys and values are read from it
                    return (
                        torch.zeros((nblk, 1, config.block_size, spec["row"]), dtype=dtype, device=self.device),
                    )
                if spec["kind"] == "state":
                    return (
                        torch.zeros(
                            (self.num_state_slots + 1, spec["width"]),
                            dtype=torch.float32,
                            device=self.device,
                        ),
                    )
                raise ValueError(f"unknown cache kind {spec['kind']!r}")

            # an entry is one spec, or a list of specs whose tensors are
            # handed to the layer together (paged rows plus a state row)
            for spec in self.model.cache_specs():
                parts = spec if isinstance(spec, (list, tuple)) else [spec]
                self.kv_caches.append(tuple(t for p in parts for t in make(p)))
        else:
            shape = (nblk, kvh, config.block_size, mc.head_dim)
            self.kv_caches: List[Tuple[torch.Tensor, torch.Tensor]] = [
                (
                    torch.zeros(shape, dtype=dtype, device=self.device),
                    torch.zeros(shape, dtype=dtype, device=self.device),
                )
                for _ in range(mc.num_layers)
            ]
        log.info(
            "KV cache: %d blocks x %d tokens (%.1f GiB), %d state slots",
            config.num_kv_blocks,
            config.block_size,
            sum(t.numel() * t.element_size() for c in self.kv_caches for t in c) / 2**30,
            self.num_state_slots,
        )
        self.adapter_manager = None
        self.graph_runner = None
        # MoE decode is graph-safe too: decode-only batches use the dense
        # expert dispatch (static shapes, no host sync — models/mixtral.py).
        # TP engines decode EAGER by default: capturing the per-block RCCL
        # all-reduce inside a hipGraph is exactly the stream-semantics
        # surface that has never run on multi-GPU hardware (docs/scaling.md)
        # — conservative by construction for the first TP run; LIG_TP_GRAPHS=1
        # opts in once validated.
        import os as _os

        self._use_graphs = (
            self.device.type == "cuda"
            and not config.enforce_eager
            and getattr(self.model, "supports_decode_graphs", True)
            and (tp is None or _os.environ.get("LIG_TP_GRAPHS", "0") == "1")
        )
        # Mixed-step prefill/decode stream overlap — MEASURED DEAD END as a
        # default: 51.4 vs 56.5 req/s at the serving shape — the graph replay and the eager
        # prefill contend for the same CUs, so splitting the step into two
        # streams only added sync overhead; the single flat mixed batch
        # already keeps the chip full.  Kept opt-in (LIG_OVERLAP=1) for
        # shapes where decode is small vs prefill.
        self._overlap = _os.environ.get("LIG_OVERLAP", "0") == "1"
        self._decode_stream = None

    # -- batch construction ---------------------------------------------------
    def _build_batch(self, out, replay: bool = False):
        """`replay`: meta.logit_rows are those the sequences ask for, instead of
        those to sample from."""
        scheduled = out.scheduled if isinstance(out, SchedulerOutput) else out
        prefills: List[ScheduledSeq] = []
        decodes: List[ScheduledSeq] = []
        for ss in scheduled:
            (decodes if ss.num_tokens == 1 else prefills).append(ss)

        bs = self.config.block_size
        ordered = prefills + decodes
        seqs = [ss.seq for ss in ordered]
        S, n_pre = len(ordered), len(prefills)
        start = np.array([q.num_computed_tokens for q in seqs], dtype=np.int64)
        length = np.array([ss.num_tokens for ss in ordered], dtype=np.int64)
        ctx = start + length
        first = np.concatenate(([0], np.cumsum(length)))  # a sequence's first flat row
        rows, ends = first.tolist(), ctx.tolist()
        T, num_prefill_tokens = rows[-1], rows[n_pre]

        # the sequences whose last known token this step processes: every
        # decode, and prompts with their final portion
        sampled = [i for i in range(n_pre) if ends[i] == seqs[i].total_len]
        sample_seqs: List[Sequence] = [seqs[i] for i in sampled] + seqs[n_pre:]
        sample_idx: List[int] = [rows[i + 1] - 1 for i in sampled] + list(range(num_prefill_tokens, T))
        if replay:
            logit_rows = []
            for ss, base in zip(ordered, rows):
                for off in ss.logit_offsets or ():
                    if not 0 <= off < ss.num_tokens:
                        raise ValueError("wanted logit offset outside the step's tokens")
                    logit_rows.append(base + off)
        else:
            # Bucket the logits GEMM's M (ROADMAP r02 #4): sample counts
            # vary 1..max_num_seqs per mixed step — pad the gather index
            # to a multiple of 64 (repeat row 0) so the 128k-vocab GEMM
            # sees a handful of stable shapes; pad rows sliced off.
            logit_rows = list(sample_idx)
            if sample_idx and self.device.type == "cuda" and self.config.pad_batch_multiple:
                logit_rows += [sample_idx[0]] * (-len(sample_idx) % 64)

        # GEMM M-bucketing: pad the flat batch tail so every projection GEMM
        # sees M % pad_batch_multiple == 0 (few stable shapes -> hipBLASLt
        # algo reuse + tile-friendly M), where the model does not ask for less.
        # Pad rows: token 0 at position 0, K/V scattered to the scratch block
        # (same slot — racy garbage is fine there), outside both attention
        # partitions and the sample set.
        num_pad_tokens = 0
        padm = self.config.pad_batch_multiple
        mgr = getattr(self, "adapter_manager", None)
        lora_tiles = None
        if mgr is not None and any(q.lora_name for q in seqs):
            slot = {name: mgr.slot_of(name) for name in {q.lora_name for q in seqs}}
            seq_slot = np.array([slot[q.lora_name] for q in seqs], dtype=np.int32)
            # of 16 rows of an adapter, or of none
            lora_tiles = int((-(-np.bincount(seq_slot + 1, length) // 16)).sum()) if getattr(mgr, "in_layer", False) else 0
        if padm > 0 and self.device.type == "cuda" and not self.config.model.is_moe:
            if hasattr(self.model, "batch_rows"):
                num_pad_tokens = self.model.batch_rows(T, padm, lora_tiles) - T
            else:
                num_pad_tokens = -T % padm

        # token ids, positions and cache slots of the flat rows, pad rows behind
        input_ids = np.zeros(T + num_pad_tokens, dtype=np.int64)
        positions = np.zeros(T + num_pad_tokens, dtype=np.int64)
        slots = np.full(T + num_pad_tokens, self.config.num_kv_blocks * bs, dtype=np.int64)
        tok_seq = np.repeat(np.arange(S, dtype=np.int32), length)
        p_bts = [q.block_table for q in seqs[:n_pre]]
        d_bts = [q.block_table for q in seqs[n_pre:]]
        p_tab = d_tab = None
        if p_bts:
            if any(len(t) * bs < c for t, c in zip(p_bts, ends)):
                raise IndexError("a sequence has fewer cache blocks than tokens")
            r = slice(0, num_prefill_tokens)
            pack_rows([q.tokens(q.num_computed_tokens, e) for q, e in zip(seqs[:n_pre], ends)], input_ids[r])
            positions[r] = np.arange(num_prefill_tokens) - (first[:-1] - start)[tok_seq[r]]
            p_tab = table_rows(p_bts)
        if d_bts:
            d_tab = np.zeros((len(d_bts), max(len(t) for t in d_bts)), dtype=np.int32)
            pack_decodes(seqs[n_pre:], bs, input_ids[num_prefill_tokens:T], positions[num_prefill_tokens:T], d_tab)
        for tab, lo, hi in ((p_tab, 0, n_pre), (d_tab, n_pre, S)):
            if tab is not None:
                r = slice(rows[lo], rows[hi])
                pos = positions[r]
                slots[r] = tab[tok_seq[r] - lo, pos // bs].astype(np.int64) * bs + pos % bs

        # every table of the step goes to the device in one copy at the end
        dev = self.device
        fields: List[Tuple[str, np.ndarray]] = []

        def put(name: str, values) -> None:
            fields.append((name, np.asarray(values, dtype=np.int32)))

        meta = BatchMeta(
            num_prefill_tokens=num_prefill_tokens,
            num_decode_tokens=len(decodes),
            slot_mapping=None,  # these come with the upload below
            max_decode_ctx=int(ctx[n_pre:].max()) if decodes else 0,
        )
        if prefills:
            put("prefill_query_start_locs", first[: n_pre + 1])
            put("prefill_context_lens", ctx[:n_pre])
            put("prefill_block_tables", p_tab)
        if decodes:
            put("decode_block_tables", d_tab)
            put("decode_context_lens", ctx[n_pre:])
        # Per-token prefill expansion, once per step (the attention layers of
        # every transformer block reuse it; see profiles/r01_bench_kernel_stats.md).
        if prefills:
            use_mfma = self.device.type == "cuda" and self.config.model.head_dim in (64, 128)
            if getattr(self.model, "needs_seq_tables", False):
                # per-layer head sizes: the model says whether any layer runs
                # the tiled kernel; none needs the per-token expansion
                use_mfma = self.device.type == "cuda" and getattr(
                    self.model, "needs_prefill_tiles", False
                )
            if use_mfma:
                # 64-row query tiles for the MFMA flash-prefill kernel.
                tiles = (length[:n_pre] + 63) // 64
                ts = np.repeat(np.arange(n_pre), tiles)
                put("prefill_tile_seq", ts)
                put("prefill_tile_qstart", (np.arange(len(ts)) - np.repeat(np.cumsum(tiles) - tiles, tiles)) * 64)
            elif not getattr(self.model, "needs_seq_tables", False):
                put("prefill_tok_context_lens", positions[:num_prefill_tokens] + 1)
                put("prefill_tok_block_tables", p_tab[tok_seq[:num_prefill_tokens]])

        # multi-LoRA: per-token adapter slot ids (-1 = base model only)
        if lora_tiles is not None:
            lora_slots = np.full(T + num_pad_tokens, -1, dtype=np.int32)  # pad rows: base model only
            lora_slots[:T] = seq_slot[tok_seq]
            put("lora_slot_per_token", lora_slots)
            if getattr(mgr, "in_layer", False):
                # row tiles over the whole batch (lora/manager.py::build_lora_rows)
                from ..lora.manager import build_lora_rows

                for name, a in zip(("tok", "len", "slot"), build_lora_rows(lora_slots)):
                    put("lora_rows_" + name, a)
            elif self.device.type == "cuda":
                # slot-grouped SGMV units (lora/manager.py::build_lora_units)
                from ..lora.manager import build_lora_units

                order, *units = build_lora_units(lora_slots)
                if len(units[0]):
                    put("lora_order", order)
                    for name, a in zip(("t0", "len", "slot"), units):
                        put("lora_unit_" + name, a)
            # prefill tokens are sequence-contiguous: 64-token segment tiles
            # per same-slot run for the MFMA SGMV path
            on = np.flatnonzero(seq_slot[:n_pre] >= 0)
            if len(on):
                tiles = (length[on] + 63) // 64
                of = np.repeat(on, tiles)
                off = (np.arange(len(of)) - np.repeat(np.cumsum(tiles) - tiles, tiles)) * 64
                put("lora_tile_t0", first[of] + off)
                put("lora_tile_len", np.minimum(64, length[of] - off))
                put("lora_tile_slot", seq_slot[of])

        if getattr(self.model, "needs_seq_tables", False):
            # Per-token / per-sequence addressing for general-size attention
            # and recurrent layers: one block-table row and one segment per
            # scheduled sequence, prefill portions first, then decodes.
            put("seq_block_tables", table_rows(p_bts + d_bts))
            put("tok_seq", np.concatenate((tok_seq, np.full(num_pad_tokens, -1, dtype=np.int32))))
            put("seg_start", first[:-1])
            put("seg_len", length)
            put("seg_slot", [max(q.state_slot, 0) for q in seqs])
            put("seg_fresh", start == 0)
            put("seg_ctx", ctx)
            meta.max_seg_len = int(length.max()) if S else 0

        # (the rows of the logits come along: an index made from a list later on
        # would wait for everything before it)
        ids_t, pos_t, meta.slot_mapping, meta.logit_rows, *tables = upload(
            [input_ids, positions, slots, np.array(logit_rows, dtype=np.int64)] + [a for _, a in fields], dev)
        for (name, _), t in zip(fields, tables):
            setattr(meta, name, t)
        return ids_t, pos_t, meta, sample_seqs, sample_idx, ordered

    # -- one step --------------------------------------------------------------
    @torch.no_grad()
    def execute(self, out: SchedulerOutput) -> Dict[int, int]:
        """Run one mixed step; returns {seq_id: sampled_token} and advances
        num_computed_tokens for every scheduled sequence."""
        if out.is_empty:
            return {}
        if self._use_graphs and all(ss.num_tokens == 1 for ss in out.scheduled):
            with gpu_range("graph_replay"):
                res = self._execute_graph(out)
            if res is not None:
                return res
        if self._use_graphs and self._overlap:
            res = self._execute_overlapped(out)
            if res is not None:
                return res
        with gpu_range("build_batch"):
            ids, pos, meta, sample_seqs, sample_idx, ordered = self._build_batch(out)
        with gpu_range("forward"), eager_tuned():
            hidden = self.model(ids, pos, self.kv_caches, meta)
        sampled: Dict[int, int] = {}
        if sample_seqs:
            with gpu_range("sample"):
                logits = self.model.compute_logits(hidden, meta.logit_rows)[: len(sample_seqs)]
                tokens = sample_tokens(logits, sample_seqs)
            for seq, tok in zip(sample_seqs, tokens):
                sampled[seq.seq_id] = tok
        for ss in ordered:
            ss.seq.num_computed_tokens += ss.num_tokens
        return sampled

    @torch.no_grad()
    def execute_replay(self, out: SchedulerOutput) -> Dict[int, torch.Tensor]:
        """Teacher-forced step: the same batch build and model forward as
        `execute`, but nothing is sampled — returns, per sequence id, the
        fp32 logits at the offsets its ScheduledSeq asks for, and advances
        num_computed_tokens."""
        if out.is_empty:
            return {}
        with gpu_range("build_batch"):
            ids, pos, meta, _, _, ordered = self._build_batch(out, replay=True)
        with gpu_range("forward"), eager_tuned():
            hidden = self.model(ids, pos, self.kv_caches, meta)
        res: Dict[int, torch.Tensor] = {}
        if len(meta.logit_rows):
            logits = self.model.compute_logits(hidden, meta.logit_rows)
            counts = [len(ss.logit_offsets or ()) for ss in ordered]
            res = {ss.seq.seq_id: part for ss, part in zip(ordered, logits.split(counts))}
        for ss in ordered:
            ss.seq.num_computed_tokens += ss.num_tokens
        return res

    def _execute_overlapped(self, out: SchedulerOutput) -> Optional[Dict[int, int]]:
        """Mixed-step stream overlap (ROADMAP r01 #9): the decode partition
        replays its hipGraph on a side stream while the prefill chunk runs
        eager on the main stream.  Safe by construction: KV slots are
        disjoint, adapter slot weights are read-only during a step, and the
        graph owns a private LoRA workspace (metadata.lora_ws)."""
        prefills = [ss for ss in out.scheduled if ss.num_tokens > 1]
        decodes = [ss for ss in out.scheduled if ss.num_tokens == 1]
        if not prefills or not decodes:
            return None
        gr = self._ensure_graph_runner()
        if gr is None or gr.pick_size(len(decodes)) is None:
            return None
        if self._decode_stream is None:
            self._decode_stream = torch.cuda.Stream(device=self.device)
        sd = self._decode_stream
        main = torch.cuda.current_stream(self.device)
        slot_of = (
            self.adapter_manager.slot_of if self.adapter_manager is not None else None
        )
        with gpu_range("overlap_step"):
            sd.wait_stream(main)  # adapter load fences etc. ride main
            with torch.cuda.stream(sd):
                logits_d = gr.run(decodes, slot_of)
            ids, pos, meta, sample_seqs_p, sample_idx_p, _ = self._build_batch(
                prefills
            )
            with eager_tuned():
                hidden = self.model(ids, pos, self.kv_caches, meta)
            logits_p = None
            if sample_seqs_p:
                idx = torch.tensor(
                    sample_idx_p, dtype=torch.int64, device=self.device
                )
                logits_p = self.model.compute_logits(hidden, idx)
            main.wait_stream(sd)
            sampled: Dict[int, int] = {}
            if logits_p is not None:
                for seq, tok in zip(
                    sample_seqs_p, sample_tokens(logits_p, sample_seqs_p)
                ):
                    sampled[seq.seq_id] = tok
            d_seqs = [ss.seq for ss in decodes]
            for seq, tok in zip(d_seqs, sample_tokens(logits_d, d_seqs)):
                sampled[seq.seq_id] = tok
        for ss in out.scheduled:
            ss.seq.num_computed_tokens += ss.num_tokens
        return sampled

    def _ensure_graph_runner(self):
        from .graph_runner import DecodeGraphRunner

        want_lora = self.adapter_manager is not None
        if self.graph_runner is None or self.graph_runner.with_lora != want_lora:
            self.graph_runner = DecodeGraphRunner(self)
            self.graph_runner.capture(with_lora=want_lora)
        return self.graph_runner

    def _execute_graph(self, out: SchedulerOutput) -> Optional[Dict[int, int]]:
        """Decode-only fast path: one hipGraph replay for the whole step."""
        decodes = out.scheduled
        gr = self._ensure_graph_runner()
        if gr.pick_size(len(decodes)) is None:
            return None  # larger than any captured bucket: eager fallback
        slot_of = (
            self.adapter_manager.slot_of if self.adapter_manager is not None else None
        )
        logits = gr.run(decodes, slot_of)
        # what the host has to do anyway, while the GPU is at it
        seqs = [ss.seq for ss in decodes]
        ids = [seq.seq_id for seq in seqs]
        for seq in seqs:
            seq.num_computed_tokens += 1
        try:
            tokens = sample_tokens(logits, seqs)
        except BaseException:
            for seq in seqs:
                seq.num_computed_tokens -= 1
            raise
        return dict(zip(ids, tokens))
