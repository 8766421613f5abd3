"""The shared matrix kernel for single query rows at the sizes where it can go
wrong: contexts around its 32-key steps and 512-key parts, group sizes on both
sides of the low-part columns, block sizes that keep or split a lane's keys,
and the options' bounds.

Tolerance: weights enter the second product as three bf16 numbers, all of their
24 bits, results are rounded to bf16 once (8 significant bits: at most 2^-8 of
the value), sums are fp32."""

import pytest
import torch

from llm_instance_gateway_amd import ops
from llm_instance_gateway_amd.ops import torch_ref

pytestmark = pytest.mark.gpu

BF = torch.bfloat16
CTX = [1, 2, 8, 31, 32, 33, 63, 64, 65, 127, 129, 511, 513, 1000, 1056]


def _batch(ctx, G, D, bs, H, seed, pad=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(BF)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    need = [(c + bs - 1) // bs for c in ctx]
    pool = sum(need) + 3
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(seed))[: sum(need)].tolist()
    tab, at = [], 0
    for k in need:
        tab.append(perm[at : at + k] + [0] * (max(need) - k))
        at += k
    n = len(ctx)
    return dict(
        q=rnd(n + pad, H * D), k=rnd(pool, G, bs, D), v=rnd(pool, G, bs, D), tab=i32(tab), ctx=i32(ctx), rnd=rnd,
        tok_seq=i32(list(range(n)) + [-1] * pad),
        pos=torch.tensor([c - 1 for c in ctx] + [0] * pad, device="cuda"),
    )


def _check(got, b, scale, H, **kw):
    args = (b["k"].double(), b["v"].double(), b["tab"], b["tok_seq"], b["pos"], scale, H)
    f = lambda v: torch_ref.paged_attention_general(b["q"].float(), args[0].float(), v.float(), *args[2:], **kw)
    ref, mag = f(args[1]), f(args[1].abs())
    assert torch.isfinite(got.float()).all()
    # 2e-5: the reference's own fp32 scores and sums
    assert ((got.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2e-5 * mag + 1e-6).all()


@pytest.mark.parametrize("nsplits", [1, 2, 5])
@pytest.mark.parametrize(
    "D,H,G,bs", [(128, 8, 2, 16), (128, 3, 1, 6), (128, 16, 2, 8), (128, 18, 2, 16), (64, 16, 1, 32), (64, 4, 4, 2), (128, 11, 1, 5)]
)
def test_decode(D, H, G, bs, nsplits):
    b = _batch(CTX, G, D, bs, H, 3)
    got = ops.paged_attention_decode(
        b["q"].view(-1, H, D), b["k"], b["v"], b["tab"], b["ctx"], D ** -0.5, nsplits=nsplits)
    _check(got.view(len(CTX), -1), b, D ** -0.5, H)


def test_decode_empty_context():
    b = _batch([5, 40], 2, 128, 16, 8, 4)
    b["ctx"][0] = 0
    got = ops.paged_attention_decode(b["q"].view(-1, 8, 128), b["k"], b["v"], b["tab"], b["ctx"], 0.1)
    assert (got[0] == 0).all() and (got[1] != 0).any()


OPTIONS = [
    {}, dict(window=1), dict(window=64), dict(window=600), dict(window=65, softcap=5.0), dict(chunk=48),
    dict(chunk=640, temp_coef=0.3, temp_every=16.0), dict(weights="sigmoid", bias=True, window=100),
    dict(weights="sigmoid", softcap=3.0), dict(sink=True, gate="entry"), dict(sink=True, gate="head", softcap=30.0, window=40),
    dict(scale=-0.2), dict(scale=0.0, window=33), dict(temp_coef=-0.9, temp_every=8.0),
]


@pytest.mark.parametrize("opt", OPTIONS, ids=range(len(OPTIONS)))
@pytest.mark.parametrize("D,H,G,bs", [(128, 4, 2, 16), (64, 12, 1, 16), (128, 6, 2, 3)])
def test_options(opt, D, H, G, bs):
    opt = dict(opt)
    b = _batch(CTX, G, D, bs, H, 5, pad=2)
    R = b["q"].shape[0]
    scale = opt.pop("scale", D ** -0.5)
    if opt.pop("bias", False):
        opt["score_bias"] = b["rnd"](H).float()
    if opt.pop("sink", False):
        opt["sink"] = b["rnd"](H).float()
    gate = opt.pop("gate", None)
    if gate:
        wide = b["rnd"](R, H * D + H + 3)
        opt["gate"] = wide[:, 3 : 3 + (H if gate == "head" else H * D)]
        opt["gate_per_head"] = gate == "head"
    wide = torch.cat([b["rnd"](R, 8), b["q"]], dim=1)  # a column block
    got = ops.paged_attention_general(
        wide[:, 8:], b["k"], b["v"], b["tab"], b["tok_seq"], b["pos"], scale, H, **opt)
    _check(got, b, scale, H, **opt)
    assert (got[-2:] == 0).all()


@pytest.mark.parametrize("D,H,G", [(128, 32, 8), (64, 8, 4)])
def test_values_of_a_wider_row(D, H, G):
    """Values read from the head of the key rows (a latent cache)."""
    b = _batch(CTX, G, D, 16, H, 6)
    wide = b["rnd"](b["k"].shape[0], G, 16, D + 64)
    b["v"] = wide[..., :D]
    got = ops.paged_attention_general(b["q"], b["k"], b["v"], b["tab"], b["tok_seq"], b["pos"], D ** -0.5, H)
    _check(got, b, D ** -0.5, H)


def test_infinite_and_lowest_scores():
    D, H, G = 128, 4, 2
    b = _batch([70, 70], G, D, 16, H, 10)
    q = b["q"].view(2, H, D)
    q[:, :, 0] = 1.0
    blk = b["tab"]
    b["k"][blk[0, 0], 0, 3, 0] = -float("inf")
    b["k"][blk[0, 1], 0, 5, 0] = torch.finfo(BF).min
    got = ops.paged_attention_decode(q, b["k"], b["v"], b["tab"], b["ctx"], D ** -0.5)
    _check(got.view(2, -1), b, D ** -0.5, H)
    q[0, 1, 7] = float("nan")
    bad = ops.paged_attention_decode(q, b["k"], b["v"], b["tab"], b["ctx"], D ** -0.5)
    assert bad[0, 1].isnan().all()
    keep = torch.ones(2, H, dtype=torch.bool, device="cuda")
    keep[0, 1] = False
    assert torch.equal(bad[keep], got[keep])


@pytest.mark.parametrize(
    "opt", [dict(window=1), dict(window=33), dict(window=64), dict(window=600), dict(chunk=48),
            dict(weights="sigmoid", window=100)], ids=range(6))
@pytest.mark.parametrize("D,H,G,bs", [(128, 8, 2, 16), (64, 12, 1, 16), (128, 18, 2, 8), (128, 6, 2, 3)])
def test_keys_before_the_first_visible_one(opt, D, H, G, bs):
    """They may hold anything, and the blocks before may be gone."""
    b = _batch(CTX, G, D, bs, H, 11)
    k, v, tab = b["k"].clone(), b["v"].clone(), b["tab"].clone()
    used = {t for row, c in zip(b["tab"].tolist(), CTX) for t in row[: (c + bs - 1) // bs]}
    gone = next(i for i in range(k.shape[0]) if i not in used)
    k[gone], v[gone] = float("nan"), float("inf")
    for s, c in enumerate(CTX):
        first = max(0, c - opt["window"]) if "window" in opt else (c - 1) // opt["chunk"] * opt["chunk"]
        tab[s, : first // bs] = gone
        if first % bs:
            k[tab[s, first // bs], :, : first % bs], v[tab[s, first // bs], :, : first % bs] = float("nan"), float("inf")
    got = ops.paged_attention_general(b["q"], k, v, tab, b["tok_seq"], b["pos"], D ** -0.5, H, **opt)
    _check(got, b, D ** -0.5, H, **opt)


# up to 32 parts; of 9248 keys' 18 parts the last is empty (17 take 17 steps each)
LONG = [1, 500, 1030, 2600, 9248, 12512, 16384]


@pytest.mark.parametrize("nsplits", [5, 32])
@pytest.mark.parametrize("D,H,G,bs", [(128, 8, 2, 16), (64, 16, 1, 32), (128, 3, 1, 6)])
def test_many_parts(D, H, G, bs, nsplits):
    b = _batch(LONG, G, D, bs, H, 19)
    got = ops.paged_attention_decode(
        b["q"].view(-1, H, D), b["k"], b["v"], b["tab"], b["ctx"], D ** -0.5, nsplits=nsplits)
    _check(got.view(len(LONG), -1), b, D ** -0.5, H)


@pytest.mark.parametrize("opt", [dict(sink=True, gate=True), dict(weights="sigmoid", gate=True), dict(softcap=8.0, window=9000)],
                         ids=range(3))
@pytest.mark.parametrize("D,H,G", [(128, 4, 1), (64, 16, 1)])
def test_many_parts_with_options(opt, D, H, G):
    opt = dict(opt)
    b = _batch(LONG, G, D, 16, H, 20, pad=1)
    assert ops.decode_nsplits(len(LONG) + 1, G, opt.get("window", 16384)) >= 17
    if opt.pop("sink", False):
        opt["sink"] = b["rnd"](H).float()
    if opt.pop("gate", False):
        opt["gate"] = b["rnd"](len(LONG) + 1, H * D)
    got = ops.paged_attention_general(b["q"], b["k"], b["v"], b["tab"], b["tok_seq"], b["pos"], D ** -0.5, H, **opt)
    _check(got, b, D ** -0.5, H, **opt)
    assert (got[-1] == 0).all()


@pytest.mark.parametrize("nsplits", [1, 5, 32])
def test_heads_of_16(nsplits):
    H, G, D = 4, 2, 16
    for ctx in (CTX, LONG):
        b = _batch(ctx, G, D, 16, H, 13)
        b["ctx"][0] = 0
        got = ops.paged_attention_decode(
            b["q"].view(-1, H, D), b["k"], b["v"], b["tab"], b["ctx"], D ** -0.5, nsplits=nsplits)
        assert (got[0] == 0).all()
        b = dict(b, q=b["q"][1:], tab=b["tab"][1:], tok_seq=b["tok_seq"][:-1], pos=b["pos"][1:])
        _check(got[1:].reshape(len(ctx) - 1, -1), b, D ** -0.5, H)


@pytest.mark.parametrize("D", [16, 64, 128])
def test_long_walks_are_cut(D):
    H, G, ns = 4, 2, 5
    b = _batch([2600, 3], G, D, 16, H, 14)
    out = torch.empty(2, H, D, dtype=BF, device="cuda")
    parts = torch.full((2, H, ns, D + 2), 7e7, device="cuda")
    ops._load_ext().paged_attention_decode_split(
        out, b["q"].view(2, H, D), b["k"], b["v"], b["tab"], b["ctx"], parts, D ** -0.5, ns, ops._stream())
    assert (parts[0] != 7e7).all() and (parts[1] == 7e7).all()
    _check(out.view(2, -1), b, D ** -0.5, H)


@pytest.mark.parametrize("weights", ["softmax", "sigmoid"])
@pytest.mark.parametrize("cap", [30.0, 1e4, 1e6])
def test_soft_caps_keep_small_scores(cap, weights):
    """A cap far above the scores changes nothing: tanh near zero may not lose
    digits (1 - 2 / (1 + e^2x) is off by 1e-7 of the cap)."""
    D, H, G = 128, 8, 2
    b = _batch(CTX, G, D, 16, H, 15)
    got = ops.paged_attention_general(
        b["q"], b["k"], b["v"], b["tab"], b["tok_seq"], b["pos"], D ** -0.5, H, softcap=cap, weights=weights)
    _check(got, b, D ** -0.5, H, softcap=cap, weights=weights)


@pytest.mark.parametrize("H,G,bias", [(32, 8, None), (32, 2, None), (32, 8, -1.0)])
def test_weights_keep_32_bits(H, G, bias):
    """Values of one sign, so that a result is off by little more than 2^-24 of
    itself.  It then differs from the rounded exact one where that lies as close
    to the middle between two bf16 numbers, which are 2^-8 to 2^-7 apart: some 2 *
    2^-24 * 180 = 2e-5 of all.  Weights of 16 bits: 1e-4 and more."""
    D, R, ctx, bs = 128, 512, 3, 16
    b = _batch([ctx] * R, G, D, bs, H, 16)
    b["v"] = 1 + b["v"].float().abs().clamp_max(1).to(BF)
    kw = {} if bias is None else dict(weights="sigmoid", score_bias=torch.full((H,), bias, device="cuda"))
    got = ops.paged_attention_general(b["q"], b["k"], b["v"], b["tab"], b["tok_seq"], b["pos"], D ** -0.5, H, **kw)
    k, v = (b[x][b["tab"][:, 0].long(), :, :ctx].double() for x in "kv")
    s = b["q"].view(R, G, H // G, D).double() @ k.transpose(-1, -2).contiguous() * D ** -0.5
    w = s.softmax(-1) if bias is None else torch.sigmoid(s + bias)
    ref = (w @ v).view(R, -1).float().to(BF)
    assert (got != ref).double().mean().item() < 4e-5


def test_more_rows_than_a_grid_dimension_holds():
    """256 threads per (row, key/value head) reach 2^32 at 16 x 1048576."""
    R, H, G, D = 1048576 + 5, 16, 16, 64
    b = _batch([1, 1], G, D, 16, H, 18)  # one key: the result is its value
    tok_seq = torch.arange(R, dtype=torch.int32, device="cuda") % 2
    q = b["rnd"](1, H * D).expand(R, H * D).contiguous()
    want = b["v"][b["tab"][:, 0].long(), :, 0].reshape(2, H * D)
    pos = torch.zeros(R, dtype=torch.int64, device="cuda")
    for got in (
        ops.paged_attention_general(q, b["k"], b["v"], b["tab"], tok_seq, pos, D ** -0.5, H),
        ops.paged_attention_decode(
            q.view(R, H, D), b["k"], b["v"], b["tab"][tok_seq.long()].contiguous(), tok_seq * 0 + 1, D ** -0.5),
    ):
        got = got.view(R, H * D)
        assert torch.equal(got[0::2], want[:1].expand(R // 2 + 1, -1)) and torch.equal(got[1::2], want[1:].expand(R // 2, -1))


@pytest.mark.parametrize("opt", [None, {}, dict(weights="sigmoid", window=100)], ids=range(3))
@pytest.mark.parametrize("D,H,G,bs", [(128, 8, 8, 16), (128, 18, 2, 8), (64, 16, 4, 32)])
def test_many_rows_are_the_few(D, H, G, bs, opt):
    """A row's result does not depend on how many come with it (from 256 rows of
    key/value heads on, values are loaded past the caches)."""
    n = 256 // G
    b = _batch([CTX[i % len(CTX)] for i in range(n)], G, D, bs, H, 23)

    def run(to):
        if opt is None:
            return ops.paged_attention_decode(b["q"][:to].view(-1, H, D), b["k"], b["v"], b["tab"][:to].contiguous(),
                                              b["ctx"][:to].contiguous(), D ** -0.5, nsplits=2).view(to, -1)
        return ops.paged_attention_general(b["q"][:to], b["k"], b["v"], b["tab"], b["tok_seq"][:to].contiguous(),
                                           b["pos"][:to].contiguous(), D ** -0.5, H, **opt)

    many = run(n)
    _check(many, b, D ** -0.5, H, **(opt or {}))
    assert torch.equal(many[: n - 1], run(n - 1))
