"""The work this framework is timed by: engine steps of the Llama-3-8B preset
with LoRA adapters, and the hybrid families' own mixers at their layer shapes.

A case is a dict of plain values; `kind` says which path it takes.

  serve    one step of the serving engine over the whole model: `decodes`
           requests that each bring one token on top of up to `ctx` cached
           ones, and `prompts` prompt portions of about `prompt_len` tokens on
           top of `cached` cached ones; `loras` adapters of rank 16 dealt out
           in turn (0: base model).  Steps without prompts run
           ModelRunner.execute (the decode graph and sampling), the others
           ModelRunner.execute_replay, which hands out the logits.  The model
           has the preset's widths and LAYERS of its layers.
  delta    ops.gated_delta_scan over `seqs` fresh prompts of about `length`
           tokens, then over one token of each
  latent   ops.latent_attention_rows over `seqs` requests with up to `ctx`
           tokens, the last `length` of which are this step's
  window   windowed attention over paged K/V: ops.paged_attention_prefill_tiles
           for prompt portions, ops.paged_attention_general for single tokens
"""

import dataclasses
import math
import random

import torch

from llm_instance_gateway_amd import ops
from llm_instance_gateway_amd.engine import EngineConfig, LLMEngine, SamplingParams
from llm_instance_gateway_amd.engine.scheduler import ScheduledSeq, SchedulerOutput
from llm_instance_gateway_amd.engine.sequence import Sequence
from llm_instance_gateway_amd.lora.manager import AdapterManager
from llm_instance_gateway_amd.models.config import get_model_config
from llm_instance_gateway_amd.utils.tunableop import maybe_enable_tunableop

DEV = "cuda:0"
BF = torch.bfloat16
BS = 16      # tokens per cache block
RANK = 16    # of every adapter
KV_STD = 0.75  # of the cached keys and values, as the random projections give
# The depth of the repository's benchmark stacks.  bf16 rounding adds up over
# the layers: the logits of the preset's 32 are 4 % off the 64-bit ones, too far
# for two correct implementations to be told from a wrong one.
LAYERS = 8


def _serve(name, decodes=0, ctx=0, prompts=0, prompt_len=0, cached=0, loras=0):
    return {"name": name, "kind": "serve", "decodes": decodes, "ctx": ctx, "prompts": prompts, "prompt_len": prompt_len,
            "cached": cached, "loras": loras}


def listed():
    return [
        # one user, one token: the latency of a step
        _serve("decode_1", decodes=1, ctx=381),
        # a few long conversations
        _serve("decode_33_long", decodes=33, ctx=6000, loras=8),
        # the saturated engine between two admissions (bench.py's concurrency and lengths)
        _serve("decode_384", decodes=384, ctx=381, loras=32),
        # the same engine in a step that admits two prompts
        _serve("mixed_382_2", decodes=382, ctx=381, prompts=2, prompt_len=202, loras=32),
        # time to first token on an idle engine
        _serve("prompt_202", prompts=1, prompt_len=202, loras=1),
        # a step whose whole token budget is fresh prompts
        _serve("prompts_20x202", prompts=20, prompt_len=200, loras=32),
        # the second budget-sized portion of a long document
        _serve("prompt_tail_4k", prompts=1, prompt_len=4096, cached=4000),
        # Daberax's delta layers: eight prompts, then their first tokens
        {"name": "delta_8x1000", "kind": "delta", "seqs": 8, "length": 1000, "heads": 32, "kv_heads": 16},
        # Lopovik's and Garesun's shared latent rows, a decode batch and prompts
        {"name": "latent_decode_256", "kind": "latent", "seqs": 256, "ctx": 1024, "length": 1, "heads": 32, "window": 0},
        {"name": "latent_4x1000", "kind": "latent", "seqs": 4, "ctx": 1000, "length": 1000, "heads": 16, "window": 0},
        # Daberax's soft-capped window over prompts
        {"name": "window_8x1000", "kind": "window", "seqs": 8, "ctx": 1000, "length": 1000, "heads": 32, "kv_heads": 8,
         "window": 512, "weights": "softmax", "cap": 30.0},
        # Vemenex's sigmoid-weighted window over a decode batch
        {"name": "window_decode_64", "kind": "window", "seqs": 64, "ctx": 1024, "length": 1, "heads": 32, "kv_heads": 8,
         "window": 512, "weights": "sigmoid", "cap": 0.0},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of its range, ends included."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "mixed", "mixed", "prompt", "prompt", "delta", "latent", "window"])
    if kind == "decode":
        n = _log(rng, 1, 384)
        # as many cached tokens in all as the saturated engine holds
        ctx = _log(rng, 64, min(8000, 160000 // n))
        c = _serve("", decodes=n, ctx=ctx, loras=rng.choice([0, _log(rng, 1, 32)]))
    elif kind == "mixed":
        n = _log(rng, 1, 384)
        ctx = _log(rng, 64, min(8000, 160000 // n))
        p = _log(rng, 1, 8)
        c = _serve("", decodes=n, ctx=ctx, prompts=p, prompt_len=_log(rng, 8, 2048 // p), loras=rng.choice([0, _log(rng, 1, 32)]))
    elif kind == "prompt":
        p = _log(rng, 1, 24)
        n = _log(rng, 8, 3600 // p)
        c = _serve("", prompts=p, prompt_len=n, cached=rng.choice([0, 0, _log(rng, 16, 4000 // p)]),
                   loras=rng.choice([0, _log(rng, 1, 32)]))
    elif kind == "delta":
        s = _log(rng, 1, 16)
        h = rng.choice([32, 64])
        c = {"name": "", "kind": "delta", "seqs": s, "length": _log(rng, 16, 8192 // s), "heads": h, "kv_heads": h // 2}
    elif kind == "latent":
        one = rng.random() < 0.5
        s = _log(rng, 1, 256 if one else 8)
        ctx = _log(rng, 64, 4096 if one else 8192 // s)
        c = {"name": "", "kind": "latent", "seqs": s, "ctx": ctx, "length": 1 if one else min(ctx, _log(rng, 16, 8192 // s)),
             "heads": rng.choice([16, 32]), "window": rng.choice([0, 512])}
    else:
        one = rng.random() < 0.5
        s = _log(rng, 1, 256 if one else 8)
        ctx = _log(rng, 64, 4096 if one else 8192 // s)
        g = rng.choice([4, 8])
        sig = rng.random() < 0.5
        c = {"name": "", "kind": "window", "seqs": s, "ctx": ctx, "length": 1 if one else min(ctx, _log(rng, 16, 8192 // s)),
             "heads": 4 * g, "kv_heads": g, "window": 512, "weights": "sigmoid" if sig else "softmax",
             "cap": 0.0 if sig else rng.choice([0.0, 30.0])}
    del c["name"]
    return c


# -- sizes that follow from a case alone ------------------------------------------------

def _lengths(case, what, n, top, low):
    """n lengths between low * top and top, the first of them top itself."""
    r = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")) + what)
    return [top] + [max(1, int(round(top * r.uniform(low, 1.0)))) for _ in range(n - 1)]


def _portions(case):
    """[(tokens cached before this step, tokens it brings)], prompts first."""
    out = []
    if case["prompts"]:
        new = _lengths(case, "new", case["prompts"], case["prompt_len"], 0.8)
        out += [(case["cached"], max(2, n)) for n in new]
    if case["decodes"]:
        out += [(c - 1, 1) for c in _lengths(case, "ctx", case["decodes"], case["ctx"], 0.5)]
    return out


def _segments(case):
    """[(tokens of the sequence after the step, tokens it brings)]"""
    ctx = _lengths(case, "ctx", case["seqs"], case["ctx"], 0.7)
    return [(c, min(c, case["length"])) for c in ctx]


def _dims(mc):
    q, kv = mc.num_heads * mc.head_dim, mc.num_kv_heads * mc.head_dim
    h, i = mc.hidden_size, mc.intermediate_size
    return {"qkv": (h, q + 2 * kv), "o": (q, h), "gate_up": (h, 2 * i), "down": (i, h)}


def _model():
    return dataclasses.replace(get_model_config("llama3-8b"), num_layers=LAYERS)


def _generator(seed, *what):
    g = torch.Generator(device=DEV)
    g.manual_seed(random.Random(repr((int(seed),) + what)).getrandbits(62))
    return g


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


# -- engine steps --------------------------------------------------------------------------

def _plan(case, seed):
    """What the requests of the step are: (cached, new, token ids, cache blocks) each, and the pool's size."""
    r = random.Random(repr((int(seed), "plan")))
    por = _portions(case)
    need = [(c + n + BS - 1) // BS for c, n in por]
    pool = sum(need) + 8
    blocks = r.sample(range(pool), sum(need))
    out, at = [], 0
    for (c, n), k in zip(por, need):
        toks = [r.randrange(1, 128000) for _ in range(n)]
        out.append((c, n, toks, blocks[at : at + k]))
        at += k
    return out, pool


def _fill_cache(k, v, seed, layer):
    g = _generator(seed, "kv", layer)
    k.normal_(0.0, KV_STD, generator=g)
    v.normal_(0.0, KV_STD, generator=g)


def _adapters(case, seed, layer, module, fin, fout):
    g = _generator(seed, "lora", layer, module)
    a = torch.empty(case["loras"], RANK, fin, dtype=BF, device=DEV).normal_(0.0, fin ** -0.5, generator=g)
    b = torch.empty(case["loras"], fout, RANK, dtype=BF, device=DEV).normal_(0.0, 0.02, generator=g)
    return a, b


def _prepare_serve(case, seed):
    mc = _model()
    plan, pool = _plan(case, seed)
    tokens = sum(n for _, n, _, _ in plan)
    longest = max(c + n for c, n, _, _ in plan)
    maybe_enable_tunableop()  # as an engine's worker process does
    cfg = EngineConfig(
        model=mc, num_kv_blocks=pool, max_num_seqs=len(plan), max_num_batched_tokens=max(512, tokens),
        max_model_len=2048 if longest <= 2048 else 8192, max_loras=max(1, case["loras"]),
    )
    torch.manual_seed(seed)
    eng = LLMEngine(cfg, device=DEV)
    runner = eng.runner
    for layer, (k, v) in enumerate(runner.kv_caches):
        _fill_cache(k[:pool], v[:pool], seed, layer)
    names = ["lora-%d" % i for i in range(case["loras"])]
    if names:
        mgr = AdapterManager(eng, max_slots=len(names), rank=RANK)
        weights = [{} for _ in names]
        for layer in range(mc.num_layers):
            for module, (fin, fout) in _dims(mc).items():
                a, b = _adapters(case, seed, layer, module, fin, fout)
                for i, w in enumerate(weights):
                    w[(layer, module)] = (a[i], b[i])
        torch.cuda.current_stream().synchronize()  # the manager copies on a stream of its own
        for name, w in zip(names, weights):
            mgr.register_weights(name, w)
        mgr.prepare(names)
        runner.adapter_manager = mgr
    scheduled = []
    for i, (cached, new, toks, blocks) in enumerate(plan):
        seq = Sequence([0] * cached + toks, sampling=SamplingParams(max_new_tokens=64),
                       lora_name=names[i % len(names)] if names else "")
        seq.num_computed_tokens = cached
        seq.block_table = blocks
        scheduled.append(ScheduledSeq(seq, new, logit_offsets=[new - 1]))
    state = {"kind": "serve", "runner": runner, "engine": eng, "out": SchedulerOutput(scheduled=scheduled),
             "decode_only": not case["prompts"], "pool": pool}
    if state["decode_only"]:
        _run_serve(state)  # the engine captures its decode graphs in its first such step
    return state


def _run_serve(state):
    runner, out = state["runner"], state["out"]
    if state["decode_only"]:
        runner.execute(out)
        graphs, n = runner.graph_runner, len(out.scheduled)
        result = graphs.logits[graphs.pick_size(n)][:n]
    else:
        logits = runner.execute_replay(out)
        k, v = runner.kv_caches[-1]
        result = {"logits": torch.cat([logits[ss.seq.seq_id] for ss in out.scheduled]),
                  "k": k[: state["pool"]], "v": v[: state["pool"]]}
    for ss in out.scheduled:  # the same step again next time
        ss.seq.num_computed_tokens -= ss.num_tokens
    return result


@torch.no_grad()
def _exact_serve(case, seed):
    mc = _model()
    plan, pool = _plan(case, seed)
    H, G, D = mc.num_heads, mc.num_kv_heads, mc.head_dim
    torch.manual_seed(seed)

    def weight(n, k):
        return torch.empty(n, k, dtype=BF, device=DEV).uniform_(-0.02, 0.02)

    embed = weight(mc.vocab_size, mc.hidden_size)
    mats = [{m: weight(fout, fin) for m, (fin, fout) in _dims(mc).items()} for _ in range(mc.num_layers)]
    head = weight(mc.vocab_size, mc.hidden_size)
    ids = torch.tensor([t for p in plan for t in p[2]], device=DEV)
    pos = torch.tensor([c + j for c, n, _, _ in plan for j in range(n)], device=DEV)
    start = [0]
    for _, n, _, _ in plan:
        start.append(start[-1] + n)
    which = torch.tensor([i % max(1, case["loras"]) for i, p in enumerate(plan) for _ in range(p[1])], device=DEV)
    slot = torch.tensor([p[3][(p[0] + j) // BS] * BS + (p[0] + j) % BS for p in plan for j in range(p[1])], device=DEV)
    angle = pos.double()[:, None] * (mc.rope_theta ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D))
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def norm(x):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + mc.rms_norm_eps)

    def turn(x):
        a, b = x[..., : D // 2], x[..., D // 2 :]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    def project(x, layer, module):
        y = x @ mats[layer][module].double().t()
        if case["loras"]:
            fin, fout = _dims(mc)[module]
            a, b = _adapters(case, seed, layer, module, fin, fout)
            for i in range(case["loras"]):
                rows = (which == i).nonzero().squeeze(1)
                if rows.numel():
                    y[rows] += (x[rows] @ a[i].double().t()) @ b[i].double().t()
        return y

    x = embed[ids].double()
    for layer in range(mc.num_layers):
        qkv = project(norm(x), layer, "qkv")
        q, k, v = (t.view(len(ids), -1, D) for t in qkv.split([H * D, G * D, G * D], dim=-1))
        q, k = turn(q), turn(k)
        kc = torch.empty(pool, G, BS, D, dtype=BF, device=DEV)
        vc = torch.empty_like(kc)
        _fill_cache(kc, vc, seed, layer)
        o = torch.empty_like(q)
        for (c, n, _, blocks), s in zip(plan, start):
            tab = torch.tensor(blocks, device=DEV)
            past = [t[tab].permute(1, 0, 2, 3).reshape(G, -1, D)[:, :c].double() for t in (kc, vc)]
            kk, vv = (torch.cat([p, t[s : s + n].transpose(0, 1)], dim=1) for p, t in zip(past, (k, v)))
            qq = q[s : s + n].view(n, G, H // G, D).permute(1, 2, 0, 3)
            seen = torch.arange(c + n, device=DEV)[None] <= torch.arange(c, c + n, device=DEV)[:, None]
            oo = o[s : s + n].view(n, G, H // G, D)
            for g in range(G) if n > 512 else [slice(None)]:  # the scores of a long portion by themselves
                kg, vg = (kk[g], vv[g]) if n > 512 else (kk[:, None], vv[:, None])
                p = (qq[g] @ kg.transpose(-1, -2) * D ** -0.5).masked_fill_(~seen, -math.inf).softmax(-1)
                r = p @ vg
                oo[:, g] = r.transpose(0, 1) if n > 512 else r.permute(2, 0, 1, 3)
        x = x + project(o.reshape(len(ids), -1), layer, "o")
        gate, up = project(norm(x), layer, "gate_up").chunk(2, dim=-1)
        x = x + project(gate * torch.sigmoid(gate) * up, layer, "down")
        mats[layer] = None
    last = torch.tensor([s - 1 for s in start[1:]], device=DEV)
    logits = norm(x[last]) @ head.double().t()
    if not case["prompts"]:
        return logits
    kc, vc = kc.double(), vc.double()
    kc[slot // BS, :, slot % BS], vc[slot // BS, :, slot % BS] = k, v
    return {"logits": logits, "k": kc, "v": vc}


def _work_serve(case):
    mc = _model()
    por = _portions(case)
    T = sum(n for _, n in por)
    dims = _dims(mc).values()
    params = mc.num_layers * sum(a * b for a, b in dims)
    kv = 2 * mc.num_kv_heads * mc.head_dim * mc.num_layers
    used = min(case["loras"], len(por))
    lora = mc.num_layers * RANK * sum(a + b for a, b in dims)
    pairs = sum(n * c + n * (n + 1) / 2 for c, n in por)
    return {
        "bytes": 2 * params + 2 * mc.vocab_size * mc.hidden_size + 2 * T * mc.hidden_size
        + 2 * kv * (sum(c for c, _ in por) + T) + 2 * used * lora + 2 * len(por) * mc.vocab_size,
        "flops": 2 * params * T + 2 * mc.vocab_size * mc.hidden_size * len(por)
        + 4 * mc.num_heads * mc.head_dim * mc.num_layers * pairs + (2 * T * lora if used else 0),
    }


# -- gated delta rule -------------------------------------------------------------------------

DELTA_DIM = 128


def _prepare_delta(case, seed):
    h, g, d = case["heads"], case["kv_heads"], DELTA_DIM
    lens = _lengths(case, "len", case["seqs"], case["length"], 0.7)
    R, S = sum(lens), case["seqs"]
    gen = _generator(seed, "delta")

    def rows(n):
        # columns of the layer's convolved projection, and its two gate columns per head
        qkv = torch.empty(n, 2 * g * d + h * d, dtype=BF, device=DEV).normal_(generator=gen)
        ba = torch.empty(n, 2 * h, device=DEV).normal_(generator=gen)
        return qkv, ba

    starts = [sum(lens[:i]) for i in range(S)]
    return {
        "kind": "delta", "case": dict(case), "lens": lens, "prompt": rows(R), "token": rows(S),
        "rate": torch.empty(h, device=DEV).uniform_(-1.0, 1.0, generator=gen),
        "bias": torch.empty(h, device=DEV).uniform_(-5.0, -3.0, generator=gen),
        "state": torch.zeros(S + 1, ops.matrix_state_width(h, d, d), device=DEV),
        "segs": (_i32(starts), _i32(lens), _i32(list(range(S))), _i32([1] * S)),
        "one": (_i32(list(range(S))), _i32([1] * S), _i32(list(range(S))), _i32([0] * S)),
    }


def _run_delta(s):
    h, g, d = s["case"]["heads"], s["case"]["kv_heads"], DELTA_DIM
    outs = []
    for (qkv, ba), segs, longest in ((s["prompt"], s["segs"], max(s["lens"])), (s["token"], s["one"], 1)):
        outs.append(ops.gated_delta_scan(
            qkv[:, : g * d], qkv[:, g * d : 2 * g * d], qkv[:, 2 * g * d :], (ba[:, :h], ba[:, h:]), s["rate"], s["bias"],
            s["state"], *segs, h, g, d, d, q_scale=d ** -0.5, max_seg_len=longest))
    return outs


def _exact_delta(case, seed):
    s = _prepare_delta(case, seed)
    h, g, d = case["heads"], case["kv_heads"], DELTA_DIM

    def inputs(rows):
        qkv, ba = (t.double() for t in rows)
        q, k, v = qkv[:, : g * d].view(-1, g, d), qkv[:, g * d : 2 * g * d].view(-1, g, d), qkv[:, 2 * g * d :].view(-1, h, d)
        q, k = (t / (t.pow(2).sum(-1, keepdim=True) + 1e-6).sqrt() for t in (q, k))
        decay = torch.exp(-s["rate"].double().exp() * torch.log1p(torch.exp(ba[:, h:] + s["bias"].double())))
        return [t.repeat_interleave(h // g, dim=1) for t in (q * d ** -0.5, k)] + [v, decay, torch.sigmoid(ba[:, :h])]

    lens, first = s["lens"], s["segs"][0].tolist()
    S = torch.zeros(case["seqs"], h, d, d, dtype=torch.float64, device=DEV)

    def step(S, q, k, v, decay, beta):
        S = S * decay[..., None, None]
        u = beta[..., None] * (v - (k[..., None, :] @ S).squeeze(-2))
        S = S + k[..., None] * u[..., None, :]
        return S, (q[..., None, :] @ S).squeeze(-2)

    rows = inputs(s["prompt"])
    out = torch.zeros(sum(lens), h, d, dtype=torch.float64, device=DEV)
    for t in range(max(lens)):
        live = [i for i, n in enumerate(lens) if t < n]
        at = torch.tensor([first[i] + t for i in live], device=DEV)
        if len(live) == case["seqs"]:
            S, out[at] = step(S, *(r[at] for r in rows))
        else:
            S[live], out[at] = step(S[live], *(r[at] for r in rows))
    _, one = step(S, *inputs(s["token"]))
    return [out.reshape(len(out), -1), one.reshape(len(one), -1)]


def _work_delta(case):
    h, g, d = case["heads"], case["kv_heads"], DELTA_DIM
    T = sum(_lengths(case, "len", case["seqs"], case["length"], 0.7)) + case["seqs"]
    return {"bytes": T * (2 * g * d * 2 + h * d * 6 + 2 * h * 4) + 3 * case["seqs"] * h * d * d * 4, "flops": 7.0 * T * h * d * d}


# -- attention of the hybrid families: latent rows, windows ---------------------------------

LATENT_ROW, LATENT_V = 576, 512
HEAD = 128


def _paged(case, seed):
    segs = _segments(case)
    need = [(c + BS - 1) // BS for c, _ in segs]
    r = random.Random(repr((int(seed), "blocks")))
    blocks = r.sample(range(sum(need) + 8), sum(need))
    table, at = [], 0
    for k in need:
        table.append(blocks[at : at + k] + [0] * (max(need) - k))
        at += k
    starts = [sum(n for _, n in segs[:i]) for i in range(len(segs) + 1)]
    return segs, starts, table, sum(need) + 8


def _prepare_latent(case, seed):
    segs, starts, table, pool = _paged(case, seed)
    gen = _generator(seed, "latent")
    return {
        "kind": "latent", "case": dict(case),
        "q": torch.empty(starts[-1], case["heads"] * LATENT_ROW, dtype=BF, device=DEV).normal_(generator=gen),
        "cache": torch.empty(pool, 1, BS, LATENT_ROW, dtype=BF, device=DEV).normal_(generator=gen),
        "sink": torch.empty(case["heads"], device=DEV).normal_(generator=gen),
        "tables": _i32(table), "start": _i32(starts[:-1]), "len": _i32([n for _, n in segs]), "ctx": _i32([c for c, _ in segs]),
        "longest": max(n for _, n in segs), "scale": (HEAD + 64) ** -0.5,
    }


def _run_latent(s):
    c = s["case"]
    return ops.latent_attention_rows(s["q"], s["cache"], LATENT_V, s["tables"], s["start"], s["len"], s["ctx"], s["longest"],
                                     s["scale"], c["heads"], sink=s["sink"], window=c["window"])


def _prepare_window(case, seed):
    segs, starts, table, pool = _paged(case, seed)
    gen = _generator(seed, "window")
    T, H, G = starts[-1], case["heads"], case["kv_heads"]
    s = {
        "kind": "window", "case": dict(case), "decode": all(n == 1 for _, n in segs),
        "q": torch.empty(T, H * HEAD, dtype=BF, device=DEV).normal_(generator=gen),
        "k": torch.empty(pool, G, BS, HEAD, dtype=BF, device=DEV).normal_(generator=gen),
        "v": torch.empty(pool, G, BS, HEAD, dtype=BF, device=DEV).normal_(generator=gen),
        "gate": torch.empty(T, H, dtype=BF, device=DEV).normal_(generator=gen),
        "tables": _i32(table),
    }
    if case["weights"] == "sigmoid":
        s["bias"] = torch.empty(H, device=DEV).normal_(-5.0, 0.5, generator=gen)
    if s["decode"]:
        s["tok_seq"] = _i32(list(range(T)))
        s["pos"] = torch.tensor([c - 1 for c, _ in segs], device=DEV)
    else:
        tiles = [(i, q) for i, (_, n) in enumerate(segs) for q in range(0, n, 64)]
        s["tile_seq"], s["tile_q"] = _i32([i for i, _ in tiles]), _i32([q for _, q in tiles])
        s["starts"], s["ctx"] = _i32(starts), _i32([c for c, _ in segs])
    return s


def _run_window(s):
    c = s["case"]
    extra = dict(gate=s["gate"], gate_per_head=True, window=c["window"], weights=c["weights"], softcap=c["cap"],
                 score_bias=s.get("bias"))
    if s["decode"]:
        return ops.paged_attention_general(s["q"], s["k"], s["v"], s["tables"], s["tok_seq"], s["pos"], HEAD ** -0.5,
                                           c["heads"], **extra)
    return ops.paged_attention_prefill_tiles(s["q"], s["k"], s["v"], s["tables"], s["starts"], s["ctx"], s["tile_seq"],
                                             s["tile_q"], HEAD ** -0.5, c["heads"], **extra)


def _seen(c, n, window):
    p = torch.arange(c - n, c, device=DEV)[:, None]
    j = torch.arange(c, device=DEV)[None]
    return (j <= p) & (p - j < window) if window else j <= p


def _exact_latent(case, seed):
    s = _prepare_latent(case, seed)
    H = case["heads"]
    out = torch.empty(len(s["q"]), H, LATENT_V, dtype=torch.float64, device=DEV)
    at = 0
    for (c, n), tab in zip(_segments(case), s["tables"].long()):
        rows = s["cache"][tab[: (c + BS - 1) // BS]].reshape(-1, LATENT_ROW)[:c].double()
        q = s["q"][at : at + n].view(n, H, LATENT_ROW).transpose(0, 1).double()
        p = (q @ rows.t() * s["scale"]).masked_fill_(~_seen(c, n, case["window"]), -math.inf)
        p = torch.cat([p, s["sink"].double().view(H, 1, 1).expand(H, n, 1)], dim=-1).softmax(-1)[..., :-1]
        out[at : at + n] = (p @ rows[:, :LATENT_V]).transpose(0, 1)
        at += n
    return out.view(at, -1)


def _exact_window(case, seed):
    s = _prepare_window(case, seed)
    H, G = case["heads"], case["kv_heads"]
    out = torch.empty(len(s["q"]), H, HEAD, dtype=torch.float64, device=DEV)
    at = 0
    for (c, n), tab in zip(_segments(case), s["tables"].long()):
        k, v = (s[x][tab[: (c + BS - 1) // BS]].permute(1, 0, 2, 3).reshape(G, 1, -1, HEAD)[:, :, :c].double() for x in "kv")
        q = s["q"][at : at + n].view(n, G, H // G, HEAD).permute(1, 2, 0, 3).double()
        p = q @ k.transpose(-1, -2) * HEAD ** -0.5
        if case["cap"]:
            p = case["cap"] * torch.tanh(p / case["cap"])
        seen = _seen(c, n, case["window"])
        if case["weights"] == "sigmoid":
            p = torch.sigmoid(p + s["bias"].double().view(G, -1, 1, 1)).masked_fill_(~seen, 0.0)
        else:
            p = p.masked_fill_(~seen, -math.inf).softmax(-1)
        o = (p @ v).permute(2, 0, 1, 3).reshape(n, H, HEAD)
        out[at : at + n] = o * torch.sigmoid(s["gate"][at : at + n].double())[..., None]
        at += n
    return out.view(at, -1)


def _pairs(case):
    """(query, key) pairs that are seen, and keys that some query sees."""
    pairs = keys = 0
    for c, n in _segments(case):
        w = case["window"] or c
        pairs += sum(min(p + 1, w) for p in range(c - n, c))
        keys += min(c, w + n - 1)
    return pairs, keys


def _work_latent(case):
    T = sum(n for _, n in _segments(case))
    pairs, keys = _pairs(case)
    return {"bytes": 2 * T * case["heads"] * (LATENT_ROW + LATENT_V) + 2 * keys * LATENT_ROW,
            "flops": 2.0 * pairs * case["heads"] * (LATENT_ROW + LATENT_V)}


def _work_window(case):
    T = sum(n for _, n in _segments(case))
    pairs, keys = _pairs(case)
    return {"bytes": 2 * T * case["heads"] * (2 * HEAD + 1) + 4 * keys * case["kv_heads"] * HEAD,
            "flops": 4.0 * pairs * case["heads"] * HEAD}


# -- what is called ------------------------------------------------------------------------------

def prepare(case, seed):
    return {"serve": _prepare_serve, "delta": _prepare_delta, "latent": _prepare_latent, "window": _prepare_window}[
        case["kind"]](case, seed)


def run(state):
    return {"serve": _run_serve, "delta": _run_delta, "latent": _run_latent, "window": _run_window}[state["kind"]](state)


def work(case):
    return {"serve": _work_serve, "delta": _work_delta, "latent": _work_latent, "window": _work_window}[case["kind"]](case)


def exact(case, seed):
    return {"serve": _exact_serve, "delta": _exact_delta, "latent": _exact_latent, "window": _exact_window}[
        case["kind"]](case, seed)


def tolerance(case):
    if case["kind"] == "serve":
        # bf16 over LAYERS layers: the kernels and plain torch ops, each 1.4 to
        # 2 % off 64 bits, are 1.1 to 1.9 % apart (largest single value: 0.1)
        return {"rel": 0.03, "max": 0.4}
    if case["kind"] == "delta":
        # fp32 results: 6e-6 off 64 bits (largest: 6e-5)
        return {"rel": 3e-5, "max": 3e-4}
    # one rounding of the weights and of the result to bf16: 2e-3 off 64 bits (largest: 0.03)
    return {"rel": 0.008, "max": 0.12}
