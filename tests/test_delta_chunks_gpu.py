"""Chunks of the gated delta rule: lengths around a chunk's edge, an odd number
of value blocks (half of a workgroup without columns), values that no 16-byte
load may read, and a resumed state, against the token-by-token reference."""

import pytest
import torch

from llm_instance_gateway_amd import ops

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _seg(*v):
    return [torch.tensor(x, dtype=torch.int32) for x in v]


def _run(dev, x, z, rate, bias, lens, heads, kv, dim, vdim, shift, state):
    nq = kv * dim
    v = x[:, 2 * nq :]
    if shift:  # the same values from an odd place and an odd stride
        wide = torch.zeros(v.shape[0], v.shape[1] + 9, dtype=BF)
        wide[:, 3 : 3 + v.shape[1]] = v
        v = wide.to(dev)[:, 3 : 3 + v.shape[1]]
    x, z = x.to(dev), z.to(dev)
    if not shift:
        v = x[:, 2 * nq :]
    outs, done = [], [0] * len(lens)
    for part in (0, 1):  # the second call resumes
        cut = [min(n, 64 + 17) if part == 0 else n for n in lens]
        n = [c - d for c, d in zip(cut, done)]
        rows = torch.cat([torch.arange(sum(lens[:i]) + done[i], sum(lens[:i]) + cut[i]) for i in range(len(lens))])
        if len(rows) == 0:
            break
        take = rows.to(dev)
        vv = v[take]
        if shift:
            w2 = torch.zeros(len(rows), v.shape[1] + 9, dtype=BF, device=dev)
            w2[:, 3 : 3 + v.shape[1]] = vv
            vv = w2[:, 3 : 3 + v.shape[1]]
        xx, zz = x[take], z[take]
        seg = _seg([sum(n[:i]) for i in range(len(n))], n, list(range(len(n))), [1 if d == 0 else 0 for d in done])
        o = ops.gated_delta_scan(xx[:, :nq], xx[:, nq : 2 * nq], vv, (zz[:, :heads], zz[:, heads:]), rate.to(dev),
                                 bias.to(dev), state, *[s.to(dev) for s in seg], heads, kv, dim, vdim,
                                 q_scale=dim ** -0.5, max_seg_len=max(n))
        outs.append((rows, o.float().cpu()))
        done = cut
    got = torch.zeros(sum(lens), heads * vdim)
    for rows, o in outs:
        got[rows] = o
    return got


@pytest.mark.parametrize("lens", [[16], [63, 64, 65], [128, 129], [17, 200, 64]])
@pytest.mark.parametrize("heads,kv,dim,vdim", [(2, 1, 64, 136), (2, 2, 32, 64), (2, 1, 128, 192), (1, 1, 200, 128), (4, 2, 24, 64)])
def test_delta_chunks(lens, heads, kv, dim, vdim):
    g = torch.Generator().manual_seed(sum(lens) + dim)
    R = sum(lens)
    x = torch.randn(R, 2 * kv * dim + heads * vdim, generator=g).to(BF)
    z = torch.randn(R, 2 * heads, generator=g)
    rate, bias = torch.randn(heads, generator=g) * 0.5, torch.randn(heads, generator=g) - 3.0
    width = ops.matrix_state_width(heads, dim, vdim)
    want = _run("cpu", x.float(), z, rate, bias, lens, heads, kv, dim, vdim, False, torch.zeros(len(lens), width))
    got = [_run("cuda", x, z, rate, bias, lens, heads, kv, dim, vdim, shift, torch.zeros(len(lens), width, device="cuda"))
           for shift in (False, True)]
    assert torch.equal(got[0], got[1])
    # products of two halves without lo * lo lose 2^-16 of themselves; a correction goes through up to four of
    # them and 64 rows, whose errors add like a walk: 4 * 8 * 2^-16 of the largest output
    assert (got[0] - want).abs().max() <= 2.0 ** -11 * want.abs().max()


@pytest.mark.parametrize("dim", [32, 64, 128])
@pytest.mark.parametrize("vdim", [128, 192])
def test_value_blocks_in_pairs(dim, vdim):
    """Prompts that fill the chip share workgroups between value blocks, alone they do not: the same bits."""
    lens, heads, kv = [17, 200, 64, 65, 130], 32, 16
    test_delta_chunks(lens, heads, kv, dim, vdim)
    g = torch.Generator("cuda").manual_seed(dim + vdim)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, z, nq = r(sum(lens), 2 * kv * dim + heads * vdim).to(BF), r(sum(lens), 2 * heads), kv * dim
    rate, bias = r(heads) * 0.5, r(heads) - 3.0
    def run(x, z, n):
        state = torch.zeros(len(n), ops.matrix_state_width(heads, dim, vdim), device="cuda")
        seg = _seg([sum(n[:i]) for i in range(len(n))], n, list(range(len(n))), [1] * len(n))
        return ops.gated_delta_scan(x[:, :nq], x[:, nq : 2 * nq], x[:, 2 * nq :], (z[:, :heads], z[:, heads:]), rate, bias,
                                    state, *[s.cuda() for s in seg], heads, kv, dim, vdim, q_scale=dim ** -0.5,
                                    max_seg_len=max(n)), state
    got, state = run(x, z, lens)
    alone = [run(x[sum(lens[:i]) :][:n].contiguous(), z[sum(lens[:i]) :][:n].contiguous(), [n]) for i, n in enumerate(lens)]
    assert torch.equal(got, torch.cat([o for o, _ in alone])) and torch.equal(state, torch.cat([s for _, s in alone]))


@pytest.mark.parametrize("heads,kv,dim", [(8, 4, 128), (16, 16, 64), (24, 12, 128), (9, 3, 128)])
def test_heads_dealt_to_the_xcds(heads, kv, dim):
    test_delta_chunks([17, 200, 64], heads, kv, dim, 64)


@pytest.mark.parametrize("dim,least", [(32, 6), (64, 5), (96, 5), (128, 5), (192, 5), (256, 4)])
def test_workgroups_to_a_cu(dim, least):
    """The first kernel is a chain of short steps, which need each other's waves to hide."""
    assert ops._hl().lig_gated_delta_prepare_workgroups(dim) >= least
