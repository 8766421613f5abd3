"""The projection kernels against 64-bit torch, at sizes that reach every tile,
its remainders and cuts of K, and the calls that stay with the library."""

import pytest
import torch

from llm_instance_gateway_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
SIZES = [
    # (rows, outputs, columns): edges of the tiles' rows and columns
    (1, 8, 64), (5, 24, 128), (16, 4096, 4096), (16, 4104, 14336), (17, 520, 192), (33, 4096, 4096), (32, 1288, 8192),
    (48, 6144, 4096), (63, 28672, 256), (65, 8200, 3584), (97, 4096, 4096), (96, 12288, 1024), (129, 6152, 4096),
    (160, 4096, 1088), (193, 4096, 14336), (202, 28680, 128), (225, 12288, 4096), (256, 22016, 512), (255, 6144, 4096),
    (257, 1288, 8192), (384, 6144, 4096), (786, 4096, 14336), (1000, 4040, 4096), (1024, 16, 64),
    (130, 4096, 4096), (343, 6144, 8192), (241, 12296, 14336), (236, 28680, 1024), (384, 65544, 256),
    (295, 8, 3072), (758, 136, 384), (833, 168, 512), (840, 8, 1344), (930, 152, 4288), (606, 4184, 4416),
    (1023, 2456, 320), (168, 17656, 320), (197, 33128, 320), (212, 32968, 320),
    (1, 928, 6400), (19, 712, 6400), (97, 4184, 4096), (129, 16648, 2112), (130, 16632, 64), (257, 23200, 3072),
    (451, 21792, 3072),
]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_projection(M, N, K):
    g = torch.Generator("cuda").manual_seed(M * 7 + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF)
    assert ops.linear_served(M, w)
    y = torch.empty(M, N, device="cuda", dtype=BF)  # by our kernel also where `linear` goes to the library
    ops._EXT.projection(y, x, w, torch.cuda.current_stream().cuda_stream)
    with torch.no_grad():
        got, parts = ops.linear(x, w), ops.linear_parts(x, w)
    ref = x.double() @ w.double().t()
    # one rounding to 8 bits; 24-bit sums over K terms, whose errors walk
    size = (x.double().pow(2) @ w.double().pow(2).t()).sqrt()
    sums = 2.0 ** -23 * K ** 0.5 * 4 * size
    for v in (y, got):
        assert v.shape == (M, N) and v.dtype == BF
        assert ((v.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + sums).all()
    # fp32, as many as K is cut into, each by the kernel that leaves sums
    assert parts.shape == (ops._EXT.projection_plan(M, N, K)[2], M, N) and parts.dtype == torch.float32
    assert ((parts.double().sum(0) - ref).abs() <= sums).all()


def test_every_tile_is_reached():
    """Each with its whole product rounded, which a size in one part runs, and with a
    part's sums (`linear_parts` runs that kernel in one part as well)."""
    plan = ops._load_ext().projection_plan
    seen = {plan(*s) for s in SIZES}
    wide = {plan(m, n, k) for m in range(1, 1025, 5)
            for n in (8, 136, 1024, 1280, 4096, 6144, 12288, 16872, 28672, 33128, 57344, 128256)
            for k in (64, 128, 320, 512, 1024, 1344, 3072, 4096, 14336) if ops._EXT.projection_serves(m, n, k)}
    kernels = lambda plans: {(m, n, cut > 1) for m, n, cut in plans}
    assert len(kernels(wide)) == 34 and kernels(seen) >= kernels(wide)
    assert {s[2] for s in seen} >= {1, 2, 8}


# one tile of rows on weights from 2^24 entries on, which are loaded past the caches
STREAMED = [
    (3, 33136, 512), (10, 33128, 512), (22, 16384, 1024), (1, 57352, 320), (67, 16872, 1024), (97, 16872, 1024),
    (79, 33128, 512), (97, 16872, 2048), (79, 57352, 320), (79, 16872, 3072), (130, 16872, 1024), (130, 33128, 512),
    (163, 33128, 512), (163, 16872, 3072), (163, 16872, 1024), (193, 3080, 8192), (163, 28680, 1024), (193, 33128, 512),
    (193, 16872, 4096), (226, 33128, 512), (33, 28672, 4096), (202, 28672, 4096),
]


@pytest.mark.parametrize("M,N,K", STREAMED)
def test_streamed_weights(M, N, K):
    test_projection(M, N, K)


def test_every_kernel_is_reached():
    """Tiles by whether they leave sums or the rounded product and by how they load W.  A
    size in one part runs both, `linear` and `linear_parts`."""
    plan = ops._load_ext().projection_plan

    def kernels(sizes):
        out = set()
        for s in sizes:
            bm, bn, cut = plan(*s)
            streams = s[0] <= bm and s[1] * s[2] >= 1 << 24
            out |= {(bm, bn, sums, streams) for sums in ((True,) if cut > 1 else (True, False))}
        return out

    wide = [(m, n, k) for m in (*range(1, 1025, 5), 1152, 1408, 1664, 1792)
            for n in (8, 136, 1024, 1280, 3072, 4096, 6144, 8192, 12288, 16384, 16872, 28672, 33128, 57344, 128256)
            for k in (64, 128, 320, 512, 1024, 1344, 2048, 3072, 4096, 8192, 14336, 28672) if ops._EXT.projection_serves(m, n, k)]
    # 17 tiles, four ways each but 16 x 32 and 32 x 32, which are for small weights
    assert len(kernels(wide)) == 64 and kernels(SIZES + STREAMED) >= kernels(wide)


@pytest.mark.parametrize("M,N,K", [(1025, 4096, 8192), (1216, 4096, 14336), (1409, 8, 8192), (1537, 2056, 8256),
                                   (2047, 4096, 8192), (2048, 1032, 8192), (1900, 8192, 16384)])
def test_more_rows_of_long_weights(M, N, K):
    """Above 1024 rows the library's, as products of shorter weights are, where nothing
    would add up the parts that they come in, or from 1793 rows on."""
    x, w = torch.randn(M, K, device="cuda").to(BF), torch.randn(N, K, device="cuda").to(BF)
    with torch.no_grad():
        assert not ops.linear_served(M, w) and ops.linear_served(1024, w)
        want = torch.nn.functional.linear(x, w)
        assert torch.equal(ops.linear(x, w), want) and torch.equal(ops.linear_parts(x, w), want)
    with pytest.raises(RuntimeError, match="shape"):
        ops._EXT.projection(want, x, w, torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("M,N,K", [(1152, 8192, 16384), (1300, 8200, 16448), (1665, 7168, 18432), (1792, 5120, 13824)])
def test_more_rows_in_one_part(M, N, K):
    test_projection(M, N, K)
    w = torch.empty(N, K, device="cuda", dtype=BF)
    assert ops.linear_pays(M, w) and not ops.linear_served(1793, w)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 448])
@pytest.mark.parametrize("M,N", [(60, 8200), (64, 1032), (130, 16632), (136, 11136), (200, 4104), (250, 70000)])
def test_fewer_stages_than_the_ring(M, N, K):
    """Column counts around the depths of the rings: what is loaded ahead and what a step waits for differ."""
    test_projection(M, N, K)


def test_other_calls_stay_with_the_library():
    g = torch.Generator("cuda").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    w = r(64, 128).to(BF)
    for x, v in ((r(8, 128), w.float()), (r(8, 72).to(BF), r(64, 72).to(BF)), (r(8, 128).to(BF), r(12, 128).to(BF)),
                 (r(128, 8).to(BF).t(), w), (r(2, 8, 128).to(BF), w), (r(8, 128).to(BF), r(128, 64).to(BF).t()),
                 (r(0, 128).to(BF), w), (r(8 * 128 + 1).to(BF)[1:].view(8, 128), w)):
        assert torch.equal(ops.linear(x, v), torch.nn.functional.linear(x, v))
    assert not ops.linear_served(1025, w) and not ops.linear_served(512, r(28672, 64).to(BF))
    p = torch.nn.Parameter(w)
    ops.linear(r(8, 128).to(BF), p).sum().backward()
    assert p.grad is not None
    with pytest.raises(RuntimeError):
        ops.linear(r(8, 64).to(BF), w)


def test_served_is_what_linear_does():
    """A layer that leaves a norm open must know that the product comes in parts: with
    a gradient to record, under a transform or forward-mode, it comes rounded."""
    w = torch.nn.Parameter(torch.ones(64, 128, device="cuda", dtype=BF))
    x = torch.ones(8, 128, device="cuda", dtype=BF)
    seen = []

    def ask(v):
        seen.append((ops.linear_served(8, w), ops.linear_parts(x, w).dim() == 3))
        return v

    ask(None)
    with torch.no_grad():
        ask(None)
        torch.vmap(ask)(torch.zeros(2))
        with torch.autograd.forward_ad.dual_level():
            ask(None)
    assert seen == [(False, False), (True, True), (False, False), (False, False)]


def test_another_device_stays_with_the_library(monkeypatch):
    w, x = torch.ones(64, 128, device="cuda", dtype=BF), torch.ones(8, 128, device="cuda", dtype=BF)
    assert ops.linear_served(8, w)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not ops.linear_served(8, w) and ops.linear_parts(x, w).dim() == 2


@pytest.mark.parametrize("M,N,K", [(24, 57344, 1024), (256, 4096, 4096), (256, 57344, 4096), (300, 6144, 4096),
                                   (448, 6144, 4096), (1000, 4096, 4096)])
def test_slower_rounded_products_stay_with_the_library(M, N, K):
    """Sizes at which the parts pay for themselves only with a reader that adds them up."""
    x = torch.randn(M, K, device="cuda").to(BF)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).to(BF)
    with torch.no_grad():
        assert torch.equal(ops.linear(x, w), torch.nn.functional.linear(x, w))
        assert ops.linear_served(M, w) and ops.linear_parts(x, w).dim() == 3


def test_watched_products_stay_with_the_library():
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode

    class Calls(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            names.append(func.__name__)
            return func(*args, **(kwargs or {}))

    g = torch.Generator("cuda").manual_seed(4)
    w, x, z = (torch.randn(n, 128, generator=g, device="cuda").to(BF) for n in (64, 8, 8))
    want, names = torch.nn.functional.linear(z, w), []
    with torch.no_grad():
        with FlopCounterMode(display=False) as flops:
            ops.linear(x, w)
        assert flops.get_total_flops() == 2 * 8 * 64 * 128
        assert torch.equal(torch.jit.trace(lambda v: ops.linear(v, w), x)(z), want)
        with Calls():
            ops.linear(x, w)
        assert "linear" in names
        with torch.device("cuda"):
            assert ops.linear_served(8, w) and ops.linear_parts(x, w).dim() == 3


# tiles that run in another's place: in one part and in several, weights past the caches and not
OTHERS = [
    (129, 33128, 128), (129, 33128, 576), (289, 8200, 3072), (129, 16392, 3072), (225, 33128, 64), (769, 7176, 8192),
    (161, 24584, 128), (161, 24584, 1024), (897, 2056, 8192), (161, 8200, 4096), (897, 11272, 3072), (513, 3080, 14336),
    (161, 16392, 3072), (193, 33128, 64), (161, 33128, 576), (641, 7176, 8192), (161, 22536, 8192), (641, 16392, 3072),
    (385, 8200, 4096), (193, 16392, 4096), (225, 40968, 64), (225, 40968, 576), (705, 16392, 3072), (705, 3080, 14336),
    (225, 16392, 4096), (769, 16392, 3072), (257, 40968, 3072), (786, 28672, 4096),
]


@pytest.mark.parametrize("M,N,K", OTHERS)
def test_tiles_in_the_place_of_others(M, N, K):
    ext = ops._load_ext()
    assert ext.projection_runs(M, N, K) != ext.projection_plan(M, N, K)[:2]
    test_projection(M, N, K)


def test_other_tiles_are_reached():
    assert len({ops._load_ext().projection_runs(*s) for s in OTHERS}) == 9
