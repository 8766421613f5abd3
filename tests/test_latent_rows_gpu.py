"""The latent-row kernel at the edges of its pieces of 8 keys, tiles of 32 and 64
keys, row blocks and slices, on the contiguous and the general fetch path.

Tolerance: weights and results are rounded to bf16 once (8 significant bits, at
most 2^-8 each), so a result is off by at most 2^-7 of the weighted sum of |v|;
sums are fp32 (1e-5 covers them and the reference's own)."""

import math

import pytest
import torch

from llm_instance_gateway_amd import ops

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _run(segs, H, D, Dv, bs, window, nsplit, gate, seed=1, scale=None, forget=False):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    need = [(c + bs - 1) // bs for c, _ in segs]
    pool = sum(need) + 2
    perm = torch.randperm(pool, generator=torch.Generator().manual_seed(seed))[: sum(need)].tolist()
    tab, at = [], 0
    for k in need:
        tab.append(perm[at : at + k] + [0] * (max(need) - k))
        at += k
    starts = [sum(n for _, n in segs[:i]) for i in range(len(segs))]
    T = sum(n for _, n in segs)
    q, cache = rnd(T, H * D).to(BF), rnd(pool, 1, bs, D).to(BF)
    # rows past every sequence's end hold what a finished request may leave behind
    for s, (c, _) in enumerate(segs):
        if c % bs:
            cache[tab[s][need[s] - 1], 0, c % bs :] = float("nan")
    sink = rnd(H)
    gt = rnd(T, H + 1).to(BF)[:, 1:] if gate else None
    scale = (D ** -0.5) if scale is None else scale
    kept, kept_tab = cache, tab
    if forget:  # keys before the first visible one hold anything, the blocks before are gone
        cache, tab = cache.clone(), [list(t) for t in tab]
        gone = next(i for i in range(pool) if i not in perm)
        cache[gone] = float("nan")
        for s, (c, n) in enumerate(segs):
            first = max(0, c - n - window + 1)
            tab[s][: first // bs] = [gone] * (first // bs)
            if first % bs:
                cache[tab[s][first // bs], 0, : first % bs] = float("nan")
    got = ops.latent_attention_rows(
        q, cache, Dv, i32(tab), i32(starts), i32([n for _, n in segs]), i32([c for c, _ in segs]),
        max(n for _, n in segs), scale, H, sink=sink, nsplit=nsplit, gate=gt, window=window)
    for s, (c, n) in enumerate(segs):
        rows = kept[torch.tensor(kept_tab[s][: need[s]], device="cuda")].reshape(-1, D)[:c].double()
        qq = q[starts[s] : starts[s] + n].view(n, H, D).transpose(0, 1).double()
        p, j = torch.arange(c - n, c, device="cuda")[:, None], torch.arange(c, device="cuda")[None]
        hide = (j > p) | ((p - j >= window) if window else (j > p))
        sc = (qq @ rows.t() * scale).masked_fill(hide, -math.inf)
        w = torch.cat([sc, sink.double().view(H, 1, 1).expand(H, n, 1)], -1).softmax(-1)[..., :-1]
        f = torch.sigmoid(gt[starts[s] : starts[s] + n].double())[..., None] if gate else 1.0
        ref = (w @ rows[:, :Dv]).transpose(0, 1) * f
        mag = (w @ rows[:, :Dv].abs()).transpose(0, 1) * f
        o = got[starts[s] : starts[s] + n].view(n, H, Dv).double()
        assert ((o - ref).abs() <= 2.0 ** -7 * mag + 1e-5).all(), (s, c, n)


ONE = [(c, 1) for c in (1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 127, 130, 300)]
MANY = [(1, 1), (9, 9), (33, 32), (65, 2), (130, 70), (300, 5)]


@pytest.mark.parametrize("nsplit", [1, 2, 5])
@pytest.mark.parametrize("window", [0, 1, 40])
@pytest.mark.parametrize("segs,H", [(ONE, 32), (ONE, 5), (MANY, 16), (MANY, 3)], ids=["one32", "one5", "many16", "many3"])
@pytest.mark.parametrize("D,Dv,bs", [(576, 512, 16), (576, 512, 8), (320, 256, 6), (72, 64, 16)])
def test_edges(segs, H, D, Dv, bs, window, nsplit):
    _run(segs, H, D, Dv, bs, window, nsplit, gate=window == 40)


@pytest.mark.parametrize("scale", [-0.05, 0.0])
def test_scale_signs(scale):
    _run(ONE, 16, 192, 128, 16, 0, 1, gate=False, scale=scale)
    _run(MANY, 16, 192, 128, 16, 0, 2, gate=True, scale=scale)


@pytest.mark.parametrize("nsplit", [1, 2])
@pytest.mark.parametrize("window", [1, 13, 40, 70])
@pytest.mark.parametrize("segs,H", [(ONE, 32), (MANY, 16), (MANY, 3)], ids=["one32", "many16", "many3"])
@pytest.mark.parametrize("D,Dv,bs", [(576, 512, 16), (576, 512, 8), (320, 256, 6), (72, 64, 16)])
def test_keys_before_the_first_visible_one(segs, H, D, Dv, bs, window, nsplit):
    _run(segs, H, D, Dv, bs, window, nsplit, gate=False, forget=True)


@pytest.mark.parametrize("segs,H", [
    ([(1000, 1000)], 16), ([(700, 100)], 16), ([(600, 300), (520, 40)], 16), ([(1500, 1)] * 16, 32), ([(520, 1)] * 160, 32),
    ([(2000, 3), (16, 16)], 5)])
def test_chosen_slices(segs, H):
    """Two workgroups a CU or more, unless a slice had less than 128 keys or there were over 32:
    fewer round more of the weights, and the error against 64 bits grows."""
    most = -(-max(c for c, _ in segs) // 16) * 16
    rows = sum(n for _, n in segs)
    cut = ops.latent_rows_nsplit(rows, len(segs), H, most)
    blocks = (rows * H + 63) // 64 + len(segs)
    assert 1 <= cut <= 32 and most // cut >= 128
    assert cut * blocks >= 512 or cut == 32 or most // (cut + 1) < 128
    _run(segs, H, 576, 512, 16, 0, 0, False)


@pytest.mark.parametrize("count", [2, 3, 8, 15, 16, 17])
@pytest.mark.parametrize("D,Dv,H", [(576, 512, 16), (72, 56, 3), (192, 128, 80)])
def test_tiles_are_dealt_over_the_segments(D, Dv, H, count):
    """Segments of no, few and many tiles; more than 16 of them are not dealt."""
    new = [(29 * i) % 90 * (i % 4 > 0) for i in range(count)]
    _run([(n + 1 + 37 * i % 200, n) for i, n in enumerate(new)], H, D, Dv, 16, 0, 1 + count % 2, gate=count == 3)


@pytest.mark.parametrize("window", [0, 1, 300, 100000])
@pytest.mark.parametrize("D,Dv,H", [(576, 512, 16), (72, 56, 3), (192, 128, 80)])
def test_tiles_are_dealt_by_their_walks(D, Dv, H, window):
    """Few rows on long contexts among longer portions of short ones, and single tokens."""
    _run([(3000, 33), (200, 200), (40, 0), (1500, 70), (900, 1), (64, 64), (2100, 120)], H, D, Dv, 16, window, 1, gate=False)


def test_results_that_lie_8_bytes_off():
    q = torch.randn(100, 16 * 72, device="cuda").to(BF)
    cache = torch.randn(8, 1, 16, 72, device="cuda").to(BF)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    args = (q, cache, 56, i32([[3, 1, 0, 2], [4, 7, 5, 6]]), i32([0, 60]), i32([60, 40]), i32([60, 64]), 60, 0.1, 16)
    out = torch.empty(100 * 16 * 56 + 4, device="cuda", dtype=BF)[4:].view(100, -1)
    assert out.data_ptr() % 16 == 8
    assert torch.equal(ops.latent_attention_rows(*args, out=out), ops.latent_attention_rows(*args))
