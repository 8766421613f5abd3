"""Fused kernels of the Llama layer against the plain ops they stand for.

Tolerance: the same fp32 arithmetic with one rounding to bf16 (8 significant
bits: at most 2^-8 of the value; the rotation's two products may be contracted
differently, 1e-6 of their size)."""

import pytest
import torch

from llm_instance_gateway_amd import ops
from llm_instance_gateway_amd.ops import torch_ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.mark.parametrize("T", [1, 15, 16, 17, 70])
@pytest.mark.parametrize("Hq,Hkv,D,bs", [(32, 8, 128, 16), (4, 2, 64, 32), (3, 1, 192, 6), (1, 1, 128, 16)])
def test_qkv_rope_cache(T, Hq, Hkv, D, bs):
    g = torch.Generator(device="cuda").manual_seed(T)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(BF)
    qkv = rnd(T, (Hq + 2 * Hkv) * D)
    blocks = (T + bs - 1) // bs + 2
    kc, vc = rnd(blocks, Hkv, bs, D), rnd(blocks, Hkv, bs, D)
    cs = ops.build_cos_sin_cache(D, 500, 1e4, "cuda").float()
    pos = torch.randint(0, 500, (T,), device="cuda", generator=g)
    slots = torch.randperm(blocks * bs, device="cuda", generator=g)[:T]
    if T > 3:
        slots[2] = -1  # not cached
    q, k, v = qkv.float().split([Hq * D, Hkv * D, Hkv * D], dim=-1)
    qr, kr = torch_ref.rotary_embedding(pos, q, k, cs, D)
    kw, vw = kc.float(), vc.float()
    live = slots >= 0
    torch_ref.reshape_and_cache(kr[live], v[live], kw, vw, slots[live])
    got = ops.qkv_rope_cache(qkv, pos, cs, kc, vc, slots, Hq)
    assert got.is_contiguous()
    for a, b in ((got, qr), (kc, kw), (vc, vw)):
        assert ((a.float() - b).abs() <= 2.0 ** -8 * b.abs() + 1e-5).all()
    assert torch.equal(vc.float(), vw)


# -- LoRA inside the layer's kernels ------------------------------------------------------
# u keeps 16 significant bits on its way through the second product, sums are
# fp32: 2^-16 of the summed magnitudes, besides the one rounding of a result.

SLOTS = [[0], [-1], [2] * 15, [1] * 16 + [-1], [3, 0, -1, 1] * 10 + [2] * 17]


def _lora(slots, seed):
    from llm_instance_gateway_amd.lora.manager import build_lora_rows

    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    toks, ln, us = (torch.from_numpy(a).cuda() for a in build_lora_rows(slots))
    # three empty tiles behind, as a decode graph pads them
    z = torch.zeros(3, 16, dtype=torch.int32, device="cuda")
    rows = (torch.cat([toks, z]), torch.cat([ln, z[:, 0]]), torch.cat([us, z[:, 0] - 1]))
    return rnd, rows, torch.tensor(slots, device="cuda")


def _delta(u, b, slots):
    """B u and the magnitude of its terms; u fp32 [T, 16]."""
    on = (slots >= 0).float()[:, None]
    bs = b.float()[slots.clamp(min=0)]
    return torch.einsum("tor,tr->to", bs, u) * on, torch.einsum("tor,tr->to", bs.abs(), u.abs()) * on


def _pack(u, rows, parts=1):
    """[T, 16] -> [parts, tiles, 16, 16], the parts adding up to it."""
    toks, ln, _ = (r.tolist() for r in rows)
    out = torch.full((parts, len(ln), 16, 16), float("nan"), device="cuda")
    for i, n in enumerate(ln):
        out[:, i, :n] = u[toks[i][:n]] / parts
    return out


def _unpack(u, rows, T):
    toks, ln, _ = (r.tolist() for r in rows)
    out = torch.zeros(T, 16, device="cuda")
    for i, n in enumerate(ln):
        out[toks[i][:n]] = u[:, i, :n].sum(0)
    return out


def _check_u(got, x, a, slots, rows):
    """A x of the rows that have an adapter."""
    on = slots >= 0
    ref = torch.einsum("trk,tk->tr", a.float()[slots.clamp(min=0)], x.float())
    mag = torch.einsum("trk,tk->tr", a.float()[slots.clamp(min=0)].abs(), x.float().abs())
    d = (_unpack(got, rows, len(slots)) - ref).abs()
    assert (d[on] <= 2.0 ** -20 * mag[on] * x.shape[1] ** 0.5 + 1e-6).all()


@pytest.mark.parametrize("slots", SLOTS, ids=range(len(SLOTS)))
@pytest.mark.parametrize("H", [256, 1024, 3072, 4096])
def test_lora_rms_norm(slots, H, monkeypatch):
    rnd, rows, sl = _lora(slots, H)
    T = len(slots)
    x, res, w = rnd(T, H).to(BF), rnd(T, H).to(BF), (1 + 0.1 * rnd(H)).to(BF)
    a, b, u = rnd(4, 16, H).to(BF), (0.1 * rnd(4, H, 16)).to(BF), rnd(T, 16)
    ws, _, _ = ops.lora_workspace(rows, H, 32, 32)
    d, mag = _delta(u, b, sl)
    # a workgroup per tile, then strips of columns where the width has whole ones
    for limit, parts in ((0, 1), (0, 15), (0, 0), (10**6, 1), (10**6, 15), (10**6, 0)):
        monkeypatch.setattr(ops, "LORA_NORM_STRIPS_BELOW", limit)
        residual = res.clone() if parts else None
        if residual is None:
            h, u_out = ops.lora_rms_norm(x, None, w, 1e-5, rows, a_stack=a, u_out=ws)
            s, tol = x.float(), 0.0
        else:
            h, u_out = ops.lora_rms_norm(x, residual, w, 1e-5, rows, _pack(u, rows, parts), b, a, ws)
            s, tol = x.float() + res.float() + d, 2.0 ** -16 * mag + 1e-6
            assert ((residual.float() - s).abs() <= 2.0 ** -8 * s.abs() + tol).all()
        ref = s * torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5) * w.float()
        rms = s.pow(2).mean(-1, keepdim=True).sqrt()
        assert ((h.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2 * tol / rms + 1e-5).all()
        _check_u(u_out, h, a, sl, rows)


@pytest.mark.parametrize("slots", SLOTS, ids=range(len(SLOTS)))
@pytest.mark.parametrize("d", [32, 160, 1024, 1056, 3584])
def test_lora_silu_and_mul(slots, d):
    rnd, rows, sl = _lora(slots, d)
    T = len(slots)
    x, u = rnd(T, 2 * d).to(BF), rnd(T, 16)
    a, b = rnd(4, 16, d).to(BF), (0.1 * rnd(4, 2 * d, 16)).to(BF)
    _, _, u_out = ops.lora_workspace(rows, 256, 32, d)
    got = ops.lora_silu_and_mul(x, rows, _pack(u, rows, 1 if d % 64 else 3), b, a, u_out)
    dl, mag = _delta(u, b, sl)
    gate, up = (x.float() + dl).chunk(2, dim=-1)
    ref = gate * torch.sigmoid(gate) * up
    mg, mu = mag.chunk(2, dim=-1)
    # silu' is at most 1.1
    tol = 2.0 ** -16 * (1.1 * mg * up.abs() + mu * (gate * torch.sigmoid(gate)).abs()) + 1e-5 * (1 + ref.abs())
    assert ((got.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + tol).all()
    _check_u(u_out, got, a, sl, rows)


def test_lora_silu_of_many_tiles():
    test_lora_silu_and_mul([2] * 600 + [-1] * 300 + [0] * 200, 4128)  # 70 tiles of 5 strips: 4 waves a workgroup


@pytest.mark.parametrize("T", [200, 1100])  # 8 and 4 waves a workgroup
def test_lora_silu_divides(T):
    """Rows without an adapter come out as those of `silu_and_mul`, bit for bit."""
    rnd, rows, _ = _lora([-1] * T, T)
    x = (3 * rnd(T, 2 * 14336)).to(BF)
    # where e^-g overflows, or nearly; the largest and smallest numbers, and none
    edge = [-86.0, -87.0, -87.5, -88.0, -88.5, -89.0, -100.0, 100.0, 3e38, -3e38, 1e-38, -1e-38, 1e-40, 0.0, -0.0,
            float("inf"), -float("inf"), float("nan")]
    x[0, : len(edge)] = torch.tensor(edge, device="cuda").to(BF)
    x[1, :14336] = torch.linspace(-95, 95, 14336, device="cuda").to(BF)
    x[0, 14336 : 14336 + len(edge)] = 1

    def bits(t):  # every NaN the same
        return torch.where(t.isnan(), torch.tensor(1.5, device="cuda", dtype=BF), t).view(torch.int16)

    def equal(a, b):
        return torch.equal(a.isnan(), b.isnan()) and torch.equal(bits(a), bits(b))

    want = ops.silu_and_mul(x)
    assert want[0, :18].isnan().tolist() == [False] * 16 + [True] * 2
    assert equal(ops.lora_silu_and_mul(x, ops.BASE_ROWS, None, None, None, None), want)
    u, a, b = rnd(1, len(rows[1]), 16, 16), rnd(1, 16, 14336).to(BF), rnd(1, 2 * 14336, 16).to(BF)
    ws = torch.empty(14, len(rows[1]), 16, 16, device="cuda")
    assert equal(ops.lora_silu_and_mul(x, rows, u, b, a, ws), want)


@pytest.mark.parametrize("slots", SLOTS, ids=range(len(SLOTS)))
@pytest.mark.parametrize("width", [32, 288, 4096])
def test_lora_shrink(slots, width):
    rnd, rows, sl = _lora(slots, width)
    x, a = rnd(len(slots), width).to(BF), rnd(4, 16, width).to(BF)
    _, u, _ = ops.lora_workspace(rows, 256, width, 32)
    ops.lora_shrink(x, rows, a, u)
    _check_u(u, x, a, sl, rows)


@pytest.mark.parametrize("slots", SLOTS, ids=range(len(SLOTS)))
@pytest.mark.parametrize("Hq,Hkv,D,bs", [(32, 8, 128, 16), (4, 2, 64, 32), (3, 1, 128, 6)])
def test_lora_qkv_rope_cache(slots, Hq, Hkv, D, bs):
    rnd, rows, sl = _lora(slots, D)
    T, W = len(slots), (Hq + 2 * Hkv) * D
    qkv, u, b = rnd(T, W).to(BF), rnd(T, 16), (0.1 * rnd(4, W, 16)).to(BF)
    blocks = (T + bs - 1) // bs + 2
    kc, vc = rnd(blocks, Hkv, bs, D).to(BF), rnd(blocks, Hkv, bs, D).to(BF)
    cs = ops.build_cos_sin_cache(D, 500, 1e4, "cuda").float()
    pos = torch.randint(0, 500, (T,), device="cuda")
    at = torch.randperm(blocks * bs, device="cuda")[:T]
    if T > 3:
        at[2] = -1
    dl, mag = _delta(u, b, sl)
    q, k, v = (qkv.float() + dl).split([Hq * D, Hkv * D, Hkv * D], dim=-1)
    qr, kr = torch_ref.rotary_embedding(pos, q, k, cs, D)
    kw, vw = kc.float(), vc.float()
    live = at >= 0
    torch_ref.reshape_and_cache(kr[live], v[live], kw, vw, at[live])
    got = ops.lora_qkv_rope_cache(qkv, pos, cs, kc, vc, at, Hq, rows, _pack(u, rows, 1 if D == 64 else 8), b)
    tol = 2.0 ** -15 * mag.max() + 1e-5  # a rotation adds two entries' errors
    for x, y in ((got, qr), (kc, kw), (vc, vw)):
        assert ((x.float() - y).abs() <= 2.0 ** -8 * y.abs() + tol).all()


@pytest.mark.parametrize("slots", SLOTS, ids=range(len(SLOTS)))
@pytest.mark.parametrize("H,cut", [(2048, 1), (3072, 3), (4096, 8), (4096, 0)])
def test_lora_norm_open(slots, H, cut):
    """The norm that leaves its factor to the readers of the product: its own
    outputs, then the rotation and the gated silu with the factor."""
    rnd, rows, sl = _lora(slots, H + cut)
    T = len(slots)
    assert ops.lora_norm_opens(rows, T, H)
    res, w, u = rnd(T, H).to(BF), (1 + 0.1 * rnd(H)).to(BF), rnd(T, 16)
    a, b = rnd(4, 16, H).to(BF), (0.1 * rnd(4, H, 16)).to(BF)
    x = rnd(cut, T, H) if cut else rnd(T, H).to(BF)
    ws, _, wd = ops.lora_workspace(rows, H, 32, 1024)
    d, mag = _delta(u, b, sl)
    for with_res in (True, False):
        residual = res.clone() if with_res else None
        if with_res:
            h, u_out, norm = ops.lora_norm_open(x, residual, w, 1e-5, rows, _pack(u, rows, 3), b, a, ws)
            s, tol = (x.sum(0) if cut else x.float()) + res.float() + d, 2.0 ** -16 * mag + 1e-5
            assert ((residual.float() - s).abs() <= 2.0 ** -8 * s.abs() + tol).all()
        else:
            h, u_out, norm = ops.lora_norm_open(res, None, w, 1e-5, rows, a_stack=a, u_out=ws)
            s, tol = res.float(), 0.0
        assert ((h.float() - s * w.float()).abs() <= 2.0 ** -8 * (s * w.float()).abs() + 2 * tol).all()
        _check_u(u_out, h, a, sl, rows)
        f = torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5)
        # readers: `y` and B u lack f; 2^-16 of the sums of B u, 2^-18 for f itself
        y, bd = rnd(T, 2048).to(BF), (0.1 * rnd(4, 2048, 16)).to(BF)
        up = _unpack(u_out, rows, T)
        dl, m2 = _delta(up, bd, sl)
        v, vm = (y.float() + dl) * f, (2.0 ** -15 * m2 + 2.0 ** -18 * y.float().abs()) * f
        got = ops.lora_silu_and_mul(y, rows, u_out, bd, rnd(4, 16, 1024).to(BF), wd, norm)
        gate, uu = v.chunk(2, dim=-1)
        tg, tu = vm.chunk(2, dim=-1)
        ref = gate * torch.sigmoid(gate) * uu
        tol = 1.1 * tg * uu.abs() + tu * (gate * torch.sigmoid(gate)).abs() + 1e-5 * (1 + ref.abs())
        assert ((got.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + tol).all()
        # 8 query, 4 key and 4 value heads of 128, the product in parts
        kc, vc = rnd(9, 4, 16, 128).to(BF), rnd(9, 4, 16, 128).to(BF)
        cs = ops.build_cos_sin_cache(128, 500, 1e4, "cuda").float()
        pos, at = torch.arange(T, device="cuda"), torch.randperm(144, device="cuda")[:T]
        yp = rnd(2, T, 2048)
        q, k, vv = ((yp.sum(0) + dl) * f).split([1024, 512, 512], dim=-1)
        qr, kr = torch_ref.rotary_embedding(pos, q, k, cs, 128)
        kw, vw = kc.float(), vc.float()
        torch_ref.reshape_and_cache(kr, vv, kw, vw, at)
        got = ops.lora_qkv_rope_cache(yp, pos, cs, kc, vc, at, 8, rows, u_out, bd, norm)
        tol = 2.0 ** -14 * (m2 * f).max() + 2.0 ** -17 * q.abs().max() + 1e-5
        for p, r in ((got, qr), (kc, kw), (vc, vw)):
            assert ((p.float() - r).abs() <= 2.0 ** -8 * r.abs() + tol).all()


@pytest.mark.parametrize("T", [1, 16, 33])
def test_base_rows(T):
    """The same kernels without a list of tiles: every row, no adapters."""
    g = torch.Generator(device="cuda").manual_seed(T)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    H, rows = 2048, ops.BASE_ROWS
    x, res, w = rnd(3, T, H), rnd(T, H).to(BF), (1 + 0.1 * rnd(H)).to(BF)
    s, residual = x.sum(0) + res.float(), res.clone()
    h, u, norm = ops.lora_norm_open(x, residual, w, 1e-5, rows)
    assert u is None and ((residual.float() - s).abs() <= 2.0 ** -8 * s.abs() + 1e-5).all()
    assert ((h.float() - s * w.float()).abs() <= 2.0 ** -8 * (s * w.float()).abs() + 1e-5).all()
    f = torch.rsqrt(s.pow(2).mean(-1, keepdim=True) + 1e-5)
    y = rnd(T, H).to(BF)
    gate, up = (y.float() * f).chunk(2, dim=-1)
    ref = gate * torch.sigmoid(gate) * up
    got = ops.lora_silu_and_mul(y, rows, None, None, None, None, norm)
    assert ((got.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * (1 + ref.abs())).all()
    kc, vc = rnd(9, 4, 16, 128).to(BF), rnd(9, 4, 16, 128).to(BF)
    cs = ops.build_cos_sin_cache(128, 500, 1e4, "cuda").float()
    pos, at = torch.arange(T, device="cuda"), torch.randperm(144, device="cuda")[:T]
    q, k, v = (x.sum(0) * f).split([1024, 512, 512], dim=-1)
    qr, kr = torch_ref.rotary_embedding(pos, q, k, cs, 128)
    kw, vw = kc.float(), vc.float()
    torch_ref.reshape_and_cache(kr, v, kw, vw, at)
    got = ops.lora_qkv_rope_cache(x, pos, cs, kc, vc, at, 8, rows, None, None, norm)
    for p, r in ((got, qr), (kc, kw), (vc, vw)):
        assert ((p.float() - r).abs() <= 2.0 ** -8 * r.abs() + 2.0 ** -17 * q.abs().max() + 1e-5).all()


@pytest.mark.parametrize("hidden", [512, 2048])  # norms a workgroup per tile, and open
def test_engine_matches_unit_kernels(monkeypatch, hidden):
    """A whole step through the in-layer kernels beside one through the SGMV
    kernels, prompts and decodes, eager and through the decode graph."""
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.lora import manager
    from llm_instance_gateway_amd.models.config import ModelConfig

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=hidden, num_layers=3, num_heads=8, num_kv_heads=2,
                     intermediate_size=768, head_dim=64, max_position_embeddings=512)
    assert ops.lora_norm_opens(ops.BASE_ROWS, 129, hidden) == (hidden == 2048)
    outs = []
    for units in (False, True):
        monkeypatch.setattr(manager, "_TILED_SGMV", False)
        torch.manual_seed(0)
        eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=200, max_num_seqs=8, max_model_len=256), device="cuda:0")
        mgr = manager.AdapterManager(eng, max_slots=3, rank=16)
        assert mgr.in_layer
        mgr.in_layer = not units
        for i in range(3):
            mgr.register_random(f"l{i}", seed=i)
        g = torch.Generator().manual_seed(5)
        for i, n in enumerate((3, 17, 40, 64, 5)):
            eng.add_request(torch.randint(1, 500, (n,), generator=g).tolist(), SamplingParams(max_new_tokens=1),
                            lora_name=["l0", "", "l2", "l1", "l0"][i])
        logits = []
        execute = eng.runner.model.compute_logits
        monkeypatch.setattr(eng.runner.model, "compute_logits", lambda h, idx: logits.append(execute(h, idx)) or logits[-1])
        eng.step()
        first = logits[-1][:5].clone()
        seqs = [eng.add_request([7 + i] * (9 + i), SamplingParams(max_new_tokens=4), lora_name=["l2", "", "l0"][i % 3]) for i in range(5)]
        eng.step()
        for s in seqs:  # the same continuation on both sides
            s.output_token_ids[-1] = 11
        for _ in range(2):  # graph replays
            eng.step()
            for s in seqs:
                s.output_token_ids[-1] = 12
        gr = eng.runner.graph_runner
        outs.append((first, gr.logits[gr.pick_size(5)][:5].float().clone()))
    for a, b in zip(*outs):
        # two correct orders of bf16 rounding, 3 layers deep
        assert (a - b).norm() <= 0.03 * b.norm()


def _wide_steps(lora, change, prompts):
    """Logits of a prompt step and of a replayed decode step of a model wide enough
    for norms that leave their factor to the readers, and how many norms did."""
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.lora import manager
    from llm_instance_gateway_amd.models.config import ModelConfig

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=2048, num_layers=3, num_heads=16, num_kv_heads=4,
                     intermediate_size=8192, head_dim=128, max_position_embeddings=512)
    torch.manual_seed(0)
    eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=200, max_num_seqs=8, max_num_batched_tokens=512,
                                 max_model_len=256), device="cuda:0")
    model = eng.runner.model
    if lora:
        mgr = manager.AdapterManager(eng, max_slots=3, rank=16)
        assert mgr.in_layer
        for i in range(3):
            mgr.register_random(f"l{i}", seed=i)
    if change is not None:
        name, how = change
        m = getattr(model.layers[1].mlp if name == "gate_up_proj" else model.layers[1].self_attn, name)
        if how == "bias":
            g = torch.Generator(device="cuda").manual_seed(3)
            m.bias = torch.nn.Parameter(0.5 * torch.randn(m.out_features, device="cuda", generator=g).to(BF))
        else:
            m.register_forward_pre_hook(lambda mod, args: (args[0].clamp(-0.5, 0.5),))
    g = torch.Generator().manual_seed(5)
    seqs = [eng.add_request(torch.randint(1, 500, (n,), generator=g).tolist(), SamplingParams(max_new_tokens=4),
                            lora_name=["l0", "", "l2", "l1", "l0"][i] if lora else "") for i, n in enumerate(prompts)]
    logits, head, opened, norm = [], model.compute_logits, [], ops.lora_norm_open
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(model, "compute_logits", lambda h, idx: logits.append(head(h, idx)) or logits[-1])
        mp.setattr(ops, "lora_norm_open", lambda *a, **k: opened.append(1) or norm(*a, **k))
        eng.step()
        first, n = logits[0][: len(seqs)].clone(), len(opened)
        for s in seqs:  # the same continuation on both sides
            s.output_token_ids[-1] = 11
        eng.step()
    gr = eng.runner.graph_runner
    return first, gr.logits[gr.pick_size(len(seqs))][: len(seqs)].float().clone(), n


CHANGES = [None] + [(m, how) for m in ("gate_up_proj", "qkv_proj") for how in ("bias", "hook")]


@pytest.mark.parametrize("change", CHANGES, ids=str)
@pytest.mark.parametrize("lora", [False, True])
def test_open_norms_match_closed(monkeypatch, lora, change):
    """Norms that leave their factor to the readers beside norms that do not, also
    where a layer's projection does more than multiply: such a module gets normed rows."""
    # 310 rows: qkv, o and down by our kernels, gate_up by the library's
    for prompts in ((5,), (33,), (100, 120, 90), (3, 17, 40, 64, 5)) if change is None else ((3, 17, 40, 64, 5),):
        a, b, n = _wide_steps(lora, change, prompts)
        with monkeypatch.context() as mp:
            mp.setattr(ops, "lora_norm_opens", lambda *a: False)
            x, y, none = _wide_steps(lora, change, prompts)
        # two correct orders of bf16 rounding, 3 layers deep
        assert (a - x).norm() <= 0.03 * x.norm() and (b - y).norm() <= 0.03 * y.norm()
        # of 6 norms; without adapters a layer of products that are not all ours is closed, and so are all in 310 rows
        want = (6 if lora or sum(prompts) <= 256 else 0) if change is None else (5 if lora else 4)
        assert (n, none) == (want, 0)


@pytest.mark.parametrize("lora", [False, True])
def test_module_hooks_run(lora):
    """The fused forwards stand aside for hooks on the modules they replace."""
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.lora import manager
    from llm_instance_gateway_amd.models.config import ModelConfig

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=512, num_layers=2, num_heads=8, num_kv_heads=2,
                     intermediate_size=1024, head_dim=64, max_position_embeddings=512)
    torch.manual_seed(0)
    eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=50, max_num_seqs=2, max_model_len=256, enforce_eager=True,
                                 pad_batch_multiple=0), device="cuda:0")
    model = eng.runner.model
    if lora:
        mgr = manager.AdapterManager(eng, max_slots=1, rank=16)
        assert mgr.in_layer
        mgr.register_random("l0", seed=1)
    seq = eng.add_request([5] * 9, SamplingParams(max_new_tokens=30), lora_name="l0" if lora else "")
    eng.step()

    def step():  # one token, the same each time, and what the head reads
        seq.output_token_ids[-1] = 11
        out, execute = [], model.compute_logits
        model.compute_logits = lambda h, idx: out.append(h.float()) or execute(h, idx)
        eng.step()
        del model.compute_logits
        seq.output_token_ids.pop()
        seq.num_computed_tokens -= 1
        return out[0]

    plain = step()
    assert lora or model._row_products()
    for m in (model.layers[0], model.layers[1].self_attn, model.layers[1].mlp) + (
            () if lora else (model.layers[0].mlp.down_proj,)):
        for register in (m.register_forward_hook, m.register_forward_pre_hook):
            calls = []
            handle = register(lambda *a: calls.append(1))
            got = step()
            handle.remove()
            assert len(calls) == 1
            assert (got - plain).norm() <= 0.03 * plain.norm()  # two orders of bf16 rounding
    assert torch.equal(step(), plain)


def test_overridden_head_reaches_the_graph():
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.models.config import get_model_config
    from llm_instance_gateway_amd.models.llama import LlamaForCausalLM

    class Negated(LlamaForCausalLM):
        def compute_logits(self, hidden, indices):
            return -super().compute_logits(hidden, indices)

    logits = []
    for cls in (LlamaForCausalLM, Negated):
        torch.manual_seed(0)
        eng = LLMEngine(EngineConfig(model=get_model_config("tiny"), num_kv_blocks=50, max_num_seqs=2, max_model_len=256),
                        device="cuda:0")
        eng.runner.model.__class__ = cls
        seq = eng.add_request([5] * 9, SamplingParams(max_new_tokens=4))
        eng.step()
        seq.output_token_ids[-1] = 11
        eng.step()
        logits.append(eng.runner.graph_runner.logits[1][:1].float().clone())
        assert seq.output_token_ids[-1] == int(logits[-1].argmax())
    assert torch.equal(logits[1], -logits[0])


@pytest.mark.parametrize("lora", [False, True])
def test_hooks_are_captured(lora):
    """What a forward hook does to a module's output is part of the decode graph."""
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.lora import manager
    from llm_instance_gateway_amd.models.config import ModelConfig

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=512, num_layers=2, num_heads=8, num_kv_heads=2,
                     intermediate_size=1024, head_dim=64, max_position_embeddings=512)
    logits = {}
    for eager in (True, False):
        torch.manual_seed(0)
        eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=50, max_num_seqs=2, max_model_len=256,
                                     enforce_eager=eager, pad_batch_multiple=0), device="cuda:0")
        model = eng.runner.model
        model.layers[0].mlp.register_forward_hook(lambda m, a, out: -out)
        if lora:
            mgr = manager.AdapterManager(eng, max_slots=1, rank=16)
            mgr.register_random("l0", seed=1)
        seqs = [eng.add_request([5 + i] * 9, SamplingParams(max_new_tokens=30),
                                lora_name="l0" if lora and i else "") for i in range(2)]
        eng.step()
        out, head = [], model.compute_logits
        for _ in range(3):
            for i, q in enumerate(seqs):
                q.output_token_ids[-1] = 11 + i
            if eager:
                model.compute_logits = lambda h, idx: out.append(head(h, idx)) or out[-1]
            eng.step()
            if not eager:
                out.append(eng.runner.graph_runner.logits[2][:2].float().clone())
        logits[eager] = out
    for a, b in zip(logits[False], logits[True]):
        assert (a - b).norm() <= 0.03 * b.norm()  # two orders of bf16 rounding


@pytest.mark.parametrize("parts", range(1, 10))
def test_every_number_of_parts(parts):
    """Norm and rotation add up a product in any number of parts, in order: the same
    24-bit sums as torch's, rounded once; cache blocks of 16 and of 6 tokens."""
    g = torch.Generator(device="cuda").manual_seed(parts)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    T, H = 19, 2048
    x, res, w = rnd(parts, T, H), rnd(T, H).to(BF), (1 + 0.1 * rnd(H)).to(BF)
    s = x[0].clone()
    for p in x[1:]:
        s += p
    residual = res.clone()
    h, _, norm = ops.lora_norm_open(x, residual, w, 1e-5, ops.BASE_ROWS)
    assert torch.equal(residual, (s + res.float()).to(BF))
    one = ops.lora_norm_open(s[None].contiguous(), res.clone(), w, 1e-5, ops.BASE_ROWS)[0]
    assert torch.equal(h, one)
    cs = ops.build_cos_sin_cache(128, 500, 1e4, "cuda").float()
    pos, at = torch.arange(T, device="cuda") * 20, torch.randperm(144, device="cuda")[:T]
    for bs in (16, 6):
        out = []
        for y in (x, s[None].contiguous()):
            kc, vc = torch.zeros(144 // bs, 4, bs, 128, dtype=BF, device="cuda"), torch.zeros(144 // bs, 4, bs, 128, dtype=BF, device="cuda")
            q = ops.lora_qkv_rope_cache(y, pos, cs, kc, vc, at, 8, ops.BASE_ROWS, None, None, norm)
            out.append((q, kc, vc))
        for a, b in zip(*out):
            assert torch.equal(a, b)


def _one_layer(hidden, inter, heads):
    from llm_instance_gateway_amd.models.config import ModelConfig
    from llm_instance_gateway_amd.models.llama import LlamaForCausalLM

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=hidden, num_layers=1, num_heads=heads, num_kv_heads=8,
                     intermediate_size=inter, head_dim=128, max_position_embeddings=512)
    return LlamaForCausalLM(mc, "cuda:0")


@torch.no_grad()
@pytest.mark.parametrize("hidden,inter,heads,step", [(4096, 14336, 32, 128), (3072, 8192, 24, 128), (2048, 8192, 16, 256)])
def test_rows_of_steps_by_the_library(hidden, inter, heads, step):
    """Above 1024 rows, to counts at which its products are not slower than at the tuned ones."""
    m = _one_layer(hidden, inter, heads)
    for tokens in (1025, 1152, 1153, 1550, 1600, 1921, 2048):
        assert m.batch_rows(tokens, 256) == -(-tokens // step) * step
        assert m.batch_rows(tokens, 64) == -(-tokens // 64) * 64
    assert m.batch_rows(2049, 256) == 2304


@torch.no_grad()
def test_rows_of_steps_whose_products_come_rounded():
    """Where norms and rotation cannot add up parts, qkv and o of such counts are the
    library's, and rows are added for them."""
    m = _one_layer(4096, 14336, 32)
    for tokens in (9, 130, 300, 786, 1000):
        few, opens = -(-tokens // 64) * 64 if tokens > 256 else tokens, tokens
        assert m.batch_rows(tokens, 256) == opens
        assert m.batch_rows(tokens, 256, 60) == opens  # adapters inside the layers
        assert m.batch_rows(tokens, 256, 96) == few  # of too many tiles for norms that open
        assert m.batch_rows(tokens, 256, 0) == few  # by kernels of their own
        hook = m.layers[0].register_forward_hook(lambda *a: None)
        assert m.batch_rows(tokens, 256) == m.batch_rows(tokens, 256, 60) == few
        hook.remove()


@pytest.mark.parametrize("rank,names,tiles", [(16, ["", ""], None), (16, ["a", "", "b", "a"], 2 + 1 + 2), (32, ["a", ""], 0)])
def test_rows_are_asked_for_with_the_adapters(monkeypatch, rank, names, tiles):
    from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
    from llm_instance_gateway_amd.lora import manager
    from llm_instance_gateway_amd.models.config import ModelConfig

    mc = ModelConfig(name="t", vocab_size=512, hidden_size=512, num_layers=1, num_heads=8, num_kv_heads=2,
                     intermediate_size=1024, head_dim=64, max_position_embeddings=512)
    eng = LLMEngine(EngineConfig(model=mc, num_kv_blocks=50, max_num_seqs=8, max_model_len=256), device="cuda:0")
    mgr = manager.AdapterManager(eng, max_slots=2, rank=rank)
    for n in "ab":
        mgr.register_random(n, seed=1)
    lens = {"": 3, "a": 10, "b": 17}
    for n in names:
        eng.add_request([1] * lens[n], SamplingParams(max_new_tokens=2), lora_name=n)
    model, asked = eng.runner.model, []
    monkeypatch.setattr(model, "batch_rows", lambda t, m, tiles=None: asked.append((t, m, tiles)) or 256)
    eng.step()
    assert asked == [(sum(lens[n] for n in names), 256, tiles)]
