"""Host arrays of a step: lists into numpy rows, numpy arrays to the device.

A step of 384 decodes turns some 15 000 Python integers (block tables) into
device tables.  A tensor per sequence costs 3.8 ms, numpy's own conversion row
by row 0.6, the native loop 0.1.  All tables of a step travel in one copy: each
would be a call of 10-20 us on the host while the device waits for the batch."""

from __future__ import annotations

import math
from typing import List, Sequence as Seq

import numpy as np
import torch

from .. import ops

ALIGN = 16  # bytes between arrays of one upload: the widest load of a kernel


def pack_rows(rows: Seq[List[int]], out: np.ndarray) -> None:
    """out[i, :len(rows[i])] = rows[i]; a 1-d `out` is filled with one after another."""
    ext = ops._load_ext()
    if ext is not None:
        ext.pack_rows(rows, out)
        return
    if out.ndim == 1:
        out[:] = [v for r in rows for v in r]
        return
    for i, r in enumerate(rows):
        out[i, : len(r)] = r


def pack_decodes(seqs: list, block_size: int, ids: np.ndarray, positions: np.ndarray, tables: np.ndarray) -> None:
    """The token that each sequence processes at num_computed_tokens, that
    position, and its cache blocks at the start of a row of `tables`."""
    ext = ops._load_ext()
    if ext is not None:
        ext.pack_decodes(seqs, block_size, ids, positions, tables)
        return
    positions[:] = [q.num_computed_tokens for q in seqs]
    if any(p // block_size >= len(q.block_table) for q, p in zip(seqs, positions.tolist())):
        raise IndexError("a sequence has fewer cache blocks than tokens")
    ids[:] = [q.tokens(p, p + 1)[0] for q, p in zip(seqs, positions.tolist())]
    pack_rows([q.block_table for q in seqs], tables)


def decode_slots(positions, tables, block_size: int, slots, context) -> None:
    """slots[i], the cache slot of row i's position by its row of `tables`;
    context[i], that position + 1."""
    ext = ops._load_ext()
    if ext is not None:
        ext.decode_slots(positions, tables, block_size, slots, context)
        return
    at = positions // block_size
    slots[:] = tables[np.arange(len(positions)), at].astype(np.int64) * block_size + positions - at * block_size
    context[:] = positions + 1


def decode_lora_rows(seqs: list, slot_of, rows: int, toks, length, slot) -> None:
    """`lora.manager.build_lora_rows` of a decode bucket: row i is sequence i,
    rows past them have no adapter; places past the last tile are empty tiles."""
    ext = ops._load_ext()
    if ext is not None:
        ext.decode_lora_rows(seqs, slot_of, rows, toks, length, slot)
        return
    from ..lora.manager import build_lora_rows

    of = {name: slot_of(name) if name and slot_of is not None else -1 for name in {q.lora_name for q in seqs}}
    slots = np.full(rows, -1, dtype=np.int32)
    slots[: len(seqs)] = [of[q.lora_name] for q in seqs]
    tok, n, s = build_lora_rows(slots)
    u = len(n)
    toks[:u], length[:u], slot[:u] = tok, n, s
    toks[u:], length[u:], slot[u:] = 0, 0, -1


def table_rows(rows: Seq[List[int]]) -> np.ndarray:
    """int32 [len(rows), longest], zero past a row's end."""
    out = np.zeros((len(rows), max(len(r) for r in rows)), dtype=np.int32)
    pack_rows(rows, out)
    return out


def lay_out(shapes) -> tuple:
    """([byte offset per (dtype, shape)], total bytes)"""
    at, offsets = 0, []
    for dtype, shape in shapes:
        offsets.append(at)
        at += -(-math.prod(shape) * _SIZE[dtype] // ALIGN) * ALIGN
    return offsets, at


_SIZE = {torch.int32: 4, torch.int64: 8}


def device_view(buf: torch.Tensor, offset: int, dtype, shape) -> torch.Tensor:
    """`shape` of int32 or int64 at a byte offset of the uint8 `buf`."""
    n = math.prod(shape) * _SIZE[dtype]
    return buf[offset : offset + n].view(dtype).view(tuple(shape))


def upload(arrays: List[np.ndarray], device: torch.device) -> List[torch.Tensor]:
    """The arrays (int32 or int64) on the device, in one copy."""
    at, places = 0, []  # in int32 places
    for a in arrays:
        places.append(at)
        at += -(-a.nbytes // ALIGN) * (ALIGN // 4)
    # the caching host allocator gives a pinned block back only after its copy
    host = torch.empty(max(at, 4), dtype=torch.int32, pin_memory=device.type == "cuda")
    h32 = host.numpy()
    h64 = h32.view(np.int64)
    for a, o in zip(arrays, places):
        if a.itemsize == 8:
            h64[o // 2 : o // 2 + a.size] = a.reshape(-1)
        else:
            h32[o : o + a.size] = a.reshape(-1)
    d32 = host.to(device, non_blocking=True)
    d64 = d32.view(torch.int64)
    out = []
    for a, o in zip(arrays, places):
        t = d64[o // 2 : o // 2 + a.size] if a.itemsize == 8 else d32[o : o + a.size]
        out.append(t if a.ndim == 1 else t.view(a.shape))
    return out
