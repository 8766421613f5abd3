"""Projections of a single token against fp32 torch: with and without the norm,
the residual and the activation, at widths of one and several batches of loads
and at row counts that leave waves and workgroups partly idle."""

import pytest
import torch

from llm_instance_gateway_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rnd(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _norm(s, w):
    return s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5) * w.float()


@pytest.mark.parametrize("K", [512, 1024, 2048, 2560, 4096, 8192])
@pytest.mark.parametrize("N", [2, 10, 96, 1030, 16390])
def test_row_product(N, K):
    g = torch.Generator("cuda").manual_seed(N + K)
    x, res = _rnd(g, 1, K).to(BF), _rnd(g, 1, K).to(BF)
    w, nw = (_rnd(g, N, K) * K ** -0.5).to(BF), (1 + 0.1 * _rnd(g, K)).to(BF)
    mag = w.float().abs() @ torch.ones(K, device="cuda")
    for norm, residual in ((None, None), (nw, None), (nw, res)):
        for silu in (False, True) if norm is not None else (False,):
            assert ops.row_product_serves(w, norm is not None)
            got = ops.row_product(x, w, norm, 1e-5, residual, silu)
            s = x.float() if residual is None else x.float() + res.float()
            if residual is not None:
                got, r = got
                assert torch.equal(r, s.to(BF))
            h = s if norm is None else _norm(s, nw)
            y = (w.float() @ h[0])
            # h is rounded to 8 bits (2^-8 of each term, like a walk), y too
            walk = 2.0 ** -8 * (w.float() ** 2 @ h[0] ** 2).sqrt() * 4 if norm is not None else 2.0 ** -18 * mag
            tol = walk + 2.0 ** -8 * y.abs() + 1e-6
            if silu:
                a, b, ta, tb = *y.chunk(2), *tol.chunk(2)
                y = torch.nn.functional.silu(a) * b
                # |silu'| <= 1.1
                tol = 1.1 * ta * (b.abs() + tb) + torch.nn.functional.silu(a).abs() * tb + 2.0 ** -7 * y.abs() + 1e-6
            assert got.shape == (1, len(y)) and ((got[0].float() - y).abs() <= tol).all()


def test_row_product_wide_and_refused():
    g = torch.Generator("cuda").manual_seed(1)
    for K in (14336, 16384):
        x, w = _rnd(g, 1, K).to(BF), (_rnd(g, 40, K) * K ** -0.5).to(BF)
        y = w.float() @ x[0].float()
        assert ((ops.row_product(x, w)[0].float() - y).abs() <= 2.0 ** -8 * y.abs() + 1e-3).all()
        assert not ops.row_product_serves(w, True)
    for w in (_rnd(g, 8, 520).to(BF), _rnd(g, 8, 512), _rnd(g, 8, 17 * 1024).to(BF), _rnd(g, 512, 8).to(BF).t()):
        assert not ops.row_product_serves(w, False)


def test_single_decode_matches_layer_kernels(monkeypatch):
    """A lone request's steps, replayed from the graph, against the same engine
    with the projections as products of their own."""
    from dataclasses import replace

    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.models.config import get_model_config
    from llm_instance_gateway_amd.models.llama import LlamaForCausalLM

    mc = replace(get_model_config("llama3-8b"), num_layers=3, vocab_size=1024)
    outs = []
    for row in (True, False):
        if not row:
            monkeypatch.setattr(LlamaForCausalLM, "_row_products", lambda self: False)
            monkeypatch.setattr(LlamaForCausalLM, "_open_norms", lambda self, rows: False)
        torch.manual_seed(3)
        eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=32, max_num_seqs=2, max_num_batched_tokens=256,
                                     max_model_len=256), device="cuda")
        if row:
            assert eng.runner.model._row_products()
        s = eng.add_request(list(range(7, 40)), SamplingParams(max_new_tokens=8))
        logits = []
        for i in range(4):
            eng.step()
            s.output_token_ids[-1] = 11 + i  # the same continuation on both sides
            if eng.runner.graph_runner is not None:
                logits.append(eng.runner.graph_runner.logits[1][:1].float().clone())
        outs.append(torch.cat(logits))
    # two correct orders of bf16 rounding, 3 layers deep
    assert (outs[0] - outs[1]).norm() <= 0.03 * outs[1].norm()


@pytest.mark.parametrize("D,Hq,Hkv,BS", [(64, 3, 1, 16), (128, 8, 2, 16), (128, 4, 4, 24), (192, 2, 1, 8)])
@pytest.mark.parametrize("slot", [0, 37, -1])  # of 40 and more
def test_heads_of_a_row(D, Hq, Hkv, BS, slot):
    """The product whose heads go where the rotation puts them, against the two by themselves."""
    g = torch.Generator("cuda").manual_seed(D + Hq + BS + slot)
    K, N = 1024, (Hq + 2 * Hkv) * D
    x, res = _rnd(g, 1, K).to(BF), _rnd(g, 1, K).to(BF)
    w, nw = (_rnd(g, N, K) * K ** -0.5).to(BF), (1 + 0.1 * _rnd(g, K)).to(BF)
    cs = ops.build_cos_sin_cache(D, 64, 10000.0, "cuda").float()
    pos, at = torch.tensor([29], device="cuda"), torch.tensor([slot], device="cuda")
    for residual in (None, res):
        caches = [[torch.full((5, Hkv, BS, D), 3.0, dtype=BF, device="cuda") for _ in "kv"] for _ in "ab"]
        got = ops.row_product_heads(x, w, nw, 1e-5, residual, pos, cs, *caches[0], at, Hq)
        y = ops.row_product(x, w, nw, 1e-5, residual)
        if residual is not None:
            got, r = got
            y, want_r = y
            assert torch.equal(r, want_r)
        want = ops.qkv_rope_cache(y, pos, cs, *caches[1], at, Hq)
        # one product of the two is rounded to 24 bits before it is added, either one: 2^-24
        # of it, which may cross one rounding to 8 bits
        for a, b in ((got, want), (caches[0][0], caches[1][0])):
            a, b = a.float(), b.float()
            assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6).all() and (a != b).float().mean() < 1e-2
        assert torch.equal(caches[0][1], caches[1][1])
        if slot < 0:
            assert (caches[0][0] == 3).all() and (caches[0][1] == 3).all()


@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("ctx", [1, 700, 1023, 1024, 2077])
@pytest.mark.parametrize("nsplits", [1, 2, 4, 16])
def test_parts_of_a_walk(D, ctx, nsplits):
    """A product that merges an attention's parts, against the one of the merged row: the same bits."""
    g = torch.Generator("cuda").manual_seed(D + ctx + nsplits)
    Hq, Hkv, BS = 1024 // D, 1024 // D // 4, 16
    nb = (ctx + BS - 1) // BS
    q, w = _rnd(g, 1, Hq, D).to(BF), (_rnd(g, 264, Hq * D) / 32).to(BF)
    k, v = (_rnd(g, nb, Hkv, BS, D).to(BF) for _ in "kv")
    table = torch.randperm(nb, generator=g, device="cuda").int().view(1, -1)
    args = (q, k, v, table, torch.tensor([ctx], dtype=torch.int32, device="cuda"), D ** -0.5)
    want = ops.row_product(ops.paged_attention_decode(*args, nsplits=nsplits).view(1, -1), w)
    x, parts = ops.paged_attention_decode_open(*args, nsplits=nsplits)
    assert (parts is not None) == (nsplits in (2, 4))  # above, a launch merges them
    assert torch.equal(ops.row_product(x, w, parts=parts), want)


@pytest.mark.parametrize("heads,opens", [(32, True), (33, False), (64, False)])
def test_wide_rows_come_merged(heads, opens):
    q, kv = torch.zeros(1, heads, 128, dtype=BF, device="cuda"), torch.zeros(70, heads, 16, 128, dtype=BF, device="cuda")
    table, ctx = torch.arange(70, dtype=torch.int32, device="cuda").view(1, -1), torch.tensor([1100], dtype=torch.int32, device="cuda")
    row, parts = ops.paged_attention_decode_open(q, kv, kv, table, ctx, 1.0, nsplits=4)
    assert (parts is not None) == opens and row.shape == (1, heads * 128)


def test_an_attend_of_its_own_is_called():
    """An instance's own `attend`, which its layer calls at any number of rows, for a single token too."""
    from dataclasses import replace

    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.models.config import get_model_config

    mc = replace(get_model_config("llama3-8b"), num_layers=2, vocab_size=1024)
    eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=32, max_num_seqs=2, max_num_batched_tokens=256, max_model_len=256,
                                 enforce_eager=True), device="cuda")
    model = eng.runner.model
    assert model._row_products()
    attn, rows = model.layers[1].self_attn, []
    theirs = attn.attend

    def attend(q, kv, meta):
        rows.append(len(q))
        return theirs(q, kv, meta)

    attn.attend = attend
    eng.add_request(list(range(7, 40)), SamplingParams(max_new_tokens=4))
    for _ in range(3):
        eng.step()
    assert rows == [33, 1, 1]


def test_a_walk_that_grows_into_parts(monkeypatch):
    """A lone request's steps, replayed from the graph, over the contexts at which its walk is cut in
    two for the first time, against the same engine with projections of their own."""
    from dataclasses import replace

    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.models.config import get_model_config
    from llm_instance_gateway_amd.models.llama import LlamaForCausalLM

    mc = replace(get_model_config("llama3-8b"), num_layers=3, vocab_size=1024)
    prompt = torch.randint(1, 1000, (985,), generator=torch.Generator().manual_seed(4)).tolist()
    outs, opened = [], []
    walk = ops.paged_attention_decode_open

    def watched(*args):
        out = walk(*args)
        opened.append(out[1])
        return out

    monkeypatch.setattr(ops, "paged_attention_decode_open", watched)
    for row in (True, False):
        if not row:
            monkeypatch.setattr(LlamaForCausalLM, "_row_products", lambda self: False)
            monkeypatch.setattr(LlamaForCausalLM, "_open_norms", lambda self, rows: False)
        torch.manual_seed(3)
        eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=160, max_num_seqs=2, max_num_batched_tokens=1024,
                                     max_model_len=2048), device="cuda")
        s = eng.add_request(prompt, SamplingParams(max_new_tokens=32))
        logits = []
        for i in range(16):  # contexts of 986 to 1000 behind the prompt: 32 steps of 32 keys from 993 on
            eng.step()
            s.output_token_ids[-1] = 11 + i
            if i:
                logits.append(eng.runner.graph_runner.logits[1][:1].float().clone())
        assert eng.runner.graph_runner._graph_nsplits(1) == 4
        outs.append(torch.cat(logits))
        # captured once, with room for parts
        assert not row or (opened and all(p is not None and p[2] == 4 for p in opened))
    # two correct orders of bf16 rounding, 3 layers deep
    assert ((outs[0] - outs[1]).norm(dim=1) <= 0.03 * outs[1].norm(dim=1)).all()
