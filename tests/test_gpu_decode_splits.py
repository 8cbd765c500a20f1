"""Decode launches whose wavefronts share a context in equal parts, within one
workgroup and over several whose results the reduce kernel merges: contexts
of every remainder around a step (32 tokens), empty and single-token ones
beside long ones, against float64 attention; and the same launches with no
workspace, which stay within one workgroup."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
ATOL = 2.0 ** -7  # bf16 probabilities and outputs, of the largest |v|


def case(seed, hq, hkv, d, ctx, fp8):
    g = torch.Generator().manual_seed(seed)
    blocks = [(c + 15) // 16 for c in ctx]
    nb = sum(blocks) + 2
    perm = torch.randperm(nb, generator=g).tolist()
    width = max(max(blocks), 1)
    bt = torch.full((len(ctx), width), -1, dtype=torch.int32)
    o = 0
    for b, n in enumerate(blocks):
        bt[b, :n] = torch.tensor(perm[o:o + n], dtype=torch.int32)
        o += n
    k = (torch.randn(nb, hkv, 16, d, generator=g) * 0.7).to(torch.bfloat16)
    v = torch.randn(nb, hkv, d, 16, generator=g).to(torch.bfloat16)
    if fp8:
        def code(t):
            c = t.float().to(torch.float8_e4m3fn).view(torch.uint8)
            return torch.where(t.float().abs() < 2.0 ** -6, torch.zeros_like(c), c)
        k, v = code(k), code(v)
    q = torch.randn(len(ctx), hq, d, generator=g).to(torch.bfloat16)
    return q, k, v, bt


def reference(q, k, v, bt, ctx):
    if k.dtype == torch.uint8:
        k, v = (t.view(torch.float8_e4m3fn).float() for t in (k, v))
    b, hq, d = q.shape
    g = hq // k.shape[1]
    out = torch.zeros(q.shape, dtype=torch.float64)
    for s, n in enumerate(ctx):
        if n == 0:
            continue
        ids = bt[s, :(n + 15) // 16].long()
        kk = k[ids].transpose(0, 1).reshape(k.shape[1], -1, d)[:, :n].double()
        vv = v[ids].permute(1, 0, 3, 2).reshape(k.shape[1], -1, d)[:, :n].double()
        for h in range(hq):
            w = torch.softmax(kk[h // g] @ q[s, h].double() / math.sqrt(d), 0)
            out[s, h] = w @ vv[h // g]
    return out


CONTEXTS = [
    [2000],                                  # several workgroups
    [0, 1, 2047, 33, 1024],                  # empty and tiny beside long
    [31, 32, 33, 63, 64, 65, 255, 257, 511, 513, 1023, 1500],
    [8000, 17, 4100],                        # FP8: more than eight partitions
    [700] * 3 + [1, 0],
    [16 * i + 5 for i in range(1, 41)],      # one workgroup each
]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (14, 2, 64), (4, 4, 128), (8, 1, 256)])
@pytest.mark.parametrize("i", range(len(CONTEXTS)))
def test_shares(pa, i, hq, hkv, d, fp8):
    ctx = CONTEXTS[i]
    q, k, v, bt = case(i, hq, hkv, d, ctx, fp8)
    ref = reference(q, k, v, bt, ctx)
    cd = torch.tensor(ctx, dtype=torch.int32).cuda()
    qd, kd, vd, btd = (t.cuda() for t in (q, k, v, bt))
    top = (v.view(torch.float8_e4m3fn) if fp8 else v).float().abs().max().item()
    out = pa.decode(qd, kd, vd, btd, cd, max(ctx))
    err = (out.cpu().double() - ref).abs().max().item()
    assert err <= ATOL * top, err
    if fp8:
        flags = torch.zeros(kd.shape[0], dtype=torch.uint8, device="cuda")
        assert torch.equal(out, pa.decode(qd, kd, vd, btd, cd, max(ctx), block_flags=flags))
    if fp8 or max(ctx) <= 2048 and d <= 128:
        # no workspace: the wavefronts of one workgroup share each context
        none = torch.empty(1, dtype=torch.uint8, device="cuda")
        alone = pa.decode(qd, kd, vd, btd, cd, max(ctx), workspace=none)
        err = (alone.cpu().double() - ref).abs().max().item()
        assert err <= ATOL * top, err


@pytest.mark.parametrize("fp8", [False, True])
def test_repeats_are_identical(pa, fp8):
    q, k, v, bt = case(3, 32, 8, 128, [1900, 400], fp8)
    args = [t.cuda() for t in (q, k, v, bt)] + [torch.tensor([1900, 400], dtype=torch.int32).cuda()]
    first = pa.decode(*args, 1900)
    for _ in range(5):
        assert torch.equal(first, pa.decode(*args, 1900))
