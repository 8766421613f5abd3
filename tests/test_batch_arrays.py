"""Host arrays of a step against the plain per-token construction."""

import numpy as np
import pytest
import torch

from llm_instance_gateway_amd import ops
from llm_instance_gateway_amd.engine import batch_arrays as ba
from llm_instance_gateway_amd.engine.sequence import Sequence

CPU = torch.device("cpu")


@pytest.fixture(params=["native", "numpy"])
def path(request, monkeypatch):
    if request.param == "numpy":
        monkeypatch.setattr(ops, "_load_ext", lambda: None)
    elif ops._load_ext() is None:
        pytest.skip("extension not built")


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_pack_rows(path, dtype):
    rows = [[3, 1, 2**31 - 1], [], [7], [np.int64(5), -1, 0, 9]]
    out = np.full((5, 4), -7, dtype=dtype)
    ba.pack_rows(rows, out)
    assert out.tolist() == [[3, 1, 2**31 - 1, -7], [-7] * 4, [7, -7, -7, -7], [5, -1, 0, 9], [-7] * 4]
    flat = np.zeros(8, dtype=dtype)
    ba.pack_rows(rows, flat)
    assert flat.tolist() == [3, 1, 2**31 - 1, 7, 5, -1, 0, 9]
    assert ba.table_rows(rows).tolist() == [[3, 1, 2**31 - 1, 0], [0] * 4, [7, 0, 0, 0], [5, -1, 0, 9]]


@pytest.mark.parametrize("rows,shape", [
    ([[1, 2, 3]], (1, 2)), ([[1], [2]], (1, 2)), ([[1, 2]], (3,)), ([[1, 2], [3, 4]], (3,)),
    ([[2**31]], (1, 1)), ([["a"]], (1, 1)), ([5], (1, 1)),
])
def test_pack_rows_refuses(path, rows, shape):
    with pytest.raises(Exception):
        ba.pack_rows(rows, np.zeros(shape, dtype=np.int32))


def _decode(computed, blocks):
    s = Sequence([5, 6, 7])
    s.output_token_ids = [8, 9]
    s.num_computed_tokens, s.block_table = computed, blocks
    return s


def test_pack_decodes(path):
    seqs = [_decode(2, [4]), _decode(3, [1, 2**31 - 1]), _decode(4, [9, 3, 6])]  # prompt's end, outputs, spare block
    ids, pos, tab = np.zeros(3, np.int64), np.zeros(3, np.int64), np.full((3, 4), -7, np.int32)
    ba.pack_decodes(seqs, 4, ids, pos, tab)
    assert ids.tolist() == [7, 8, 9] and pos.tolist() == [2, 3, 4]
    assert tab.tolist() == [[4, -7, -7, -7], [1, 2**31 - 1, -7, -7], [9, 3, 6, -7]]


def test_pack_decodes_reads_numbers_of_any_kind(path):
    """of one digit inside, of more, negative, zero, numpy's and truth values"""
    seqs = [_decode(2, [b, 0]) for b in (2**30 - 1, 2**30, -1, 0, np.int64(6), True)]
    for s, t in zip(seqs, (2**40, -5, 0, 2**30, np.int32(3), False)):
        s.prompt_token_ids[2] = t
    ids, pos, tab = np.zeros(6, np.int64), np.zeros(6, np.int64), np.full((6, 2), -7, np.int32)
    ba.pack_decodes(seqs, 4, ids, pos, tab)
    assert tab[:, 0].tolist() == [2**30 - 1, 2**30, -1, 0, 6, 1] and ids.tolist() == [2**40, -5, 0, 2**30, 3, 0]


@pytest.mark.parametrize("computed,blocks,room", [(4, [1], 4), (2, [], 4), (5, [1, 2], 4), (2, [1, 2, 3], 2)])
def test_pack_decodes_refuses(path, computed, blocks, room):
    """too few blocks, none, no such token, more blocks than room"""
    with pytest.raises(Exception):
        ba.pack_decodes([_decode(computed, blocks)], 4, np.zeros(1, np.int64), np.zeros(1, np.int64),
                        np.zeros((1, room), np.int32))


@pytest.mark.parametrize("which", range(3))
def test_pack_decodes_fills_or_refuses(path, which):
    """Arrays of another type are not filled as a copy and dropped."""
    types = [np.int64, np.int64, np.int32]
    types[which] = np.int16
    ids, pos, tab = (np.zeros(shape, t) for shape, t in zip((1, 1, (1, 2)), types))
    try:
        ba.pack_decodes([_decode(3, [6])], 4, ids, pos, tab)
    except TypeError:
        return
    assert (ids.tolist(), pos.tolist(), tab.tolist()) == ([8], [3], [[6, 0]])


def test_decode_slots(path):
    pos, tab = np.array([0, 7, 4, 11]), np.array([[3, 0, 0], [1, 2**31 - 1, 0], [5, 6, 0], [0, 0, 9]], np.int32)
    slots, ctx = np.zeros(4, np.int64), np.zeros(4, np.int32)
    ba.decode_slots(pos, tab, 4, slots, ctx)
    assert slots.tolist() == [12, (2**31 - 1) * 4 + 3, 24, 39] and ctx.tolist() == [1, 8, 5, 12]
    with pytest.raises(IndexError):
        ba.decode_slots(pos + 8, tab, 4, slots, ctx)


@pytest.mark.parametrize("names,rows", [([], 3), (["a"], 1), (["b", "", "a", "b", "x"], 8), (["a"] * 33 + [""] * 5 + ["b"] * 16, 64),
                                        (["ab"[i % 2] for i in range(40)], 40)])
def test_decode_lora_rows(path, names, rows):
    from llm_instance_gateway_amd.lora.manager import build_lora_rows, max_lora_rows

    asked = []
    slot_of = lambda name: asked.append(name) or {"a": 4, "b": 0}.get(name, -1)
    seqs = [Sequence([1], lora_name=n) for n in names]
    room = max_lora_rows(rows, 6)
    tok, n, slot = (np.full(s, -7, np.int32) for s in ((room, 16), room, room))
    ba.decode_lora_rows(seqs, slot_of, rows, tok, n, slot)
    want = build_lora_rows(np.array([{"a": 4, "b": 0}.get(x, -1) for x in names] + [-1] * (rows - len(names)), dtype=np.int32))
    u = len(want[1])
    for got, w in zip((tok, n, slot), want):
        assert got[:u].tolist() == w.tolist()
    assert not tok[u:].any() and not n[u:].any() and (slot[u:] == -1).all()
    assert sorted(asked) == sorted({x for x in names if x})  # each name once, "" never


def test_upload_keeps_values_and_alignment():
    arrays = [np.arange(3, dtype=np.int64), np.zeros((0, 4), np.int32), np.arange(10, dtype=np.int32).reshape(5, 2),
              np.arange(12, dtype=np.int32).reshape(3, 4).T, np.array([9], dtype=np.int64)]
    got = ba.upload(arrays, CPU)
    for a, t in zip(arrays, got):
        assert t.numpy().dtype == a.dtype and t.tolist() == a.tolist() and t.is_contiguous()
        assert (t.data_ptr() - got[0].data_ptr()) % ba.ALIGN == 0


@pytest.mark.parametrize("out", [0, 4])
def test_sequence_tokens(out):
    s = Sequence([1, 2, 3])
    s.output_token_ids = list(range(10, 10 + out))
    for a in range(3 + out + 1):
        for b in range(a, 3 + out + 1):
            assert s.tokens(a, b) == s.all_token_ids[a:b]


def test_build_batch_matches_per_token_construction():
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine
    from llm_instance_gateway_amd.engine.scheduler import ScheduledSeq
    from llm_instance_gateway_amd.models.config import get_model_config

    eng = LLMEngine(EngineConfig(model=get_model_config("tiny"), num_kv_blocks=64, max_num_seqs=8,
                                 max_num_batched_tokens=256, max_model_len=256), device="cpu")
    r, bs = eng.runner, eng.config.block_size if hasattr(eng, "config") else eng.runner.config.block_size
    blocks = iter(range(63, 0, -1))
    sched, order = [], []
    for cached, n, extra in ((0, 1, 0), (0, 5, 0), (bs, bs + 1, 3), (2 * bs - 1, 1, 0), (3, bs, 0), (bs, 1, 7)):
        s = Sequence(list(range(100, 100 + cached + n + extra)))
        s.num_computed_tokens = cached
        s.block_table = [next(blocks) for _ in range(-(-(cached + n + extra) // bs))]
        sched.append(ScheduledSeq(s, n))
    ids, pos, meta, seqs, idx, ordered = r._build_batch(sched)
    order = [x for x in sched if x.num_tokens > 1] + [x for x in sched if x.num_tokens == 1]
    assert [x.seq for x in ordered] == [x.seq for x in order]
    want = [(x.seq, p) for x in order for p in range(x.seq.num_computed_tokens, x.seq.num_computed_tokens + x.num_tokens)]
    assert ids.tolist() == [s.all_token_ids[p] for s, p in want] and pos.tolist() == [p for _, p in want]
    assert meta.slot_mapping.tolist() == [s.block_table[p // bs] * bs + p % bs for s, p in want]
    assert meta.num_prefill_tokens == 5 + bs + 1 + bs and meta.num_decode_tokens == 3
    assert meta.prefill_query_start_locs.tolist() == [0, 5, 6 + bs, 6 + 2 * bs]
    assert meta.prefill_context_lens.tolist() == [5, 2 * bs + 1, 3 + bs]
    assert meta.decode_context_lens.tolist() == [1, 2 * bs, bs + 1] and meta.max_decode_ctx == 2 * bs
    for tab, part in ((meta.prefill_block_tables, order[:3]), (meta.decode_block_tables, order[3:])):
        w = max(len(x.seq.block_table) for x in part)
        assert tab.tolist() == [x.seq.block_table + [0] * (w - len(x.seq.block_table)) for x in part]
    # a prompt's unfinished portion samples nothing, every one-token row does
    done = [i for i, x in enumerate(order) if x.num_tokens == 1 or x.seq.num_computed_tokens + x.num_tokens == x.seq.total_len]
    assert seqs == [order[i].seq for i in done]
    assert [ids[i].item() for i in idx] == [
        s.all_token_ids[x.seq.num_computed_tokens + x.num_tokens - 1] for s, x in ((order[i].seq, order[i]) for i in done)]
    sched[0].seq.block_table = []
    with pytest.raises(IndexError):
        r._build_batch(sched)
