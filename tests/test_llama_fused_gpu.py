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
