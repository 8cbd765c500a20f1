"""pa_prefill's three work splits (256, 128 and 64 query rows per workgroup, the
latter two with the keys of a tile split over two groups) at the edges of
their tiles, and the numbering of the work items over sequences: against
float64 attention over the same bf16 / FP8 values."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# Probabilities and outputs are rounded to bf16 (2^-9 each) and the
# probabilities' errors average over the keys: 2^-7 of the row's largest |v|.
ATOL = 2.0 ** -7


def attend64(q, k, v, tables, q_lens, past, nb, scale):
    """Per sequence; block ids outside [0, nb) hold no keys."""
    hq, d = q.shape[1:]
    g = hq // k.shape[1]
    out, row = torch.zeros(q.shape, dtype=torch.float64, device=q.device), 0
    for n, p, ids in zip(q_lens, past, tables):
        if n == 0:
            continue
        ctx = p + n
        idx = torch.tensor(ids[:(ctx + 15) // 16], device=q.device)
        ok = (idx >= 0) & (idx < nb)
        idx = torch.where(ok, idx, torch.zeros_like(idx))
        kk = k[idx].transpose(0, 1).reshape(k.shape[1], -1, d)[:, :ctx].double()
        vv = v[idx].permute(1, 0, 3, 2).reshape(k.shape[1], -1, d)[:, :ctx].double()
        keep = ok.repeat_interleave(16)[:ctx]
        mask = (torch.arange(ctx, device=q.device)[None] <=
                (p + torch.arange(n, device=q.device))[:, None]) & keep[None]
        for h in range(hq):
            s = q[row:row + n, h].double() @ kk[h // g].t().contiguous() * scale
            s = s.masked_fill(~mask, -math.inf)
            w = torch.nan_to_num(torch.softmax(s, -1))
            out[row:row + n, h] = w @ vv[h // g]
        row += n
    return out


def check(pa, seed, hq, hkv, d, q_lens, past, fp8=False, bad=(), shift=0.0):
    g = torch.Generator().manual_seed(seed)
    ctx = [a + b for a, b in zip(q_lens, past)]
    blocks = [(c + 15) // 16 for c in ctx]
    nb = sum(blocks) + 3
    perm = torch.randperm(nb, generator=g).tolist()
    tables, o = [], 0
    for n in blocks:
        tables.append(perm[o:o + n])
        o += n
    for s, b in bad:
        tables[s][b] = nb + 5 if b % 2 else -1
    k = torch.randn(nb, hkv, 16, d, generator=g) * 0.7 + shift
    v = torch.randn(nb, hkv, d, 16, generator=g)
    q = torch.randn(sum(q_lens), hq, d, generator=g) - shift
    q, k, v = (t.to(torch.bfloat16).cuda() for t in (q, k, v))
    if fp8:
        def code(t):
            c = t.float().clamp(-200, 200).to(torch.float8_e4m3fn).view(torch.uint8)
            return torch.where(t.float().abs() < 2.0 ** -6, torch.zeros_like(c), c)
        kc, vc = code(k), code(v)
        k, v = (c.view(torch.float8_e4m3fn).float() for c in (kc, vc))
    else:
        # stale cache entries past the contexts may hold any bits
        for n, ids in zip(ctx, tables):
            if n % 16 and 0 <= ids[-1] < nb:
                k[ids[-1], :, n % 16:] = math.nan
                v[ids[-1], :, :, n % 16:] = math.nan
        kc, vc = k, v
    width = max(blocks + [1])
    bt = torch.tensor([t + [0] * (width - len(t)) for t in tables], dtype=torch.int32).cuda()
    cu = torch.tensor([0] + torch.tensor(q_lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    pl = torch.tensor(past, dtype=torch.int32).cuda()
    scale = d ** -0.5
    out = pa.prefill(q, kc, vc, bt, cu, pl, max(q_lens), scale=scale)
    ref = attend64(q, k, v, tables, q_lens, past, nb, scale)
    top = torch.nan_to_num(v.float()).abs().max().item()
    err = (out.double() - ref).abs().max().item()
    assert err <= ATOL * top, (err, top)


EDGES = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 129]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 64), (6, 2, 128), (8, 2, 128), (14, 2, 64),
                                      (12, 3, 64), (16, 8, 128)])
def test_small_launches_at_tile_edges(pa, hq, hkv, d, fp8):
    """Few items: 64 rows per workgroup."""
    for i, n in enumerate(EDGES):
        for p in (0, 1, 31, 33, 64, 95):
            check(pa, 100 * i + p, hq, hkv, d, [n], [p], fp8)
    check(pa, 7, hq, hkv, d, EDGES, EDGES[::-1], fp8)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,d,copies", [(32, 8, 128, 12), (14, 2, 64, 30), (8, 2, 128, 30),
                                             (32, 8, 128, 40), (14, 2, 64, 110)])
def test_larger_launches(pa, hq, hkv, d, copies, fp8):
    """128, then 256 rows per workgroup, ragged, with empty sequences."""
    n = [(37 * i) % 211 for i in range(copies)] + [0, 300]
    p = [(53 * i) % 97 for i in range(copies)] + [5, 0]
    check(pa, copies, hq, hkv, d, n, p, fp8)


@pytest.mark.parametrize("seqs", [63, 64, 65, 130, 256, 257, 300])
def test_many_sequences(pa, seqs):
    """Ranks and item numbers over several rounds of 64 sequences, and past
    the sequences that are numbered through."""
    n = [1 + (i * 7) % 23 if i % 9 else 0 for i in range(seqs)]
    p = [(i * 13) % 61 for i in range(seqs)]
    check(pa, seqs, 8, 2, 64, n, p)


@pytest.mark.parametrize("hq,hkv", [(8, 2), (32, 8)])
def test_invalid_blocks_first(pa, hq, hkv):
    """Keys in blocks outside the pool are masked, also where they are all of
    a key group's first step, before scores far below zero."""
    check(pa, 3, hq, hkv, 128, [70, 5], [40, 90], bad=[(0, 0), (0, 1), (1, 2), (1, 3)], shift=1.5)
    check(pa, 4, hq, hkv, 128, [400] * 12, [0] * 12, bad=[(2, 0), (2, 1), (5, 2), (5, 3)],
          shift=1.5)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("shift", [0.0, 40.0])
@pytest.mark.parametrize("hq,hkv,d,copies", [(8, 2, 128, 1), (14, 2, 64, 1), (32, 8, 128, 12),
                                             (14, 2, 64, 30), (32, 8, 128, 40), (14, 2, 64, 110)])
def test_absent_keys_change_nothing(pa, hq, hkv, d, copies, shift, fp8):
    """A table that begins with a whole tile (64 keys) of ids outside the pool
    gives the bits of the table without them: its first present keys are
    scored as any sequence's first keys are, also far below zero (shift 40:
    scores of about -18000)."""
    g = torch.Generator().manual_seed(copies)
    q_lens = [1 + (37 * i + 69) % 211 for i in range(copies)]
    past = [(53 * i) % 97 for i in range(copies)]
    blocks = [(n + p + 15) // 16 for n, p in zip(q_lens, past)]
    nb = sum(blocks)
    k = torch.randn(nb, hkv, 16, d, generator=g) * 0.7 + shift
    v = torch.randn(nb, hkv, d, 16, generator=g)
    q = (torch.randn(sum(q_lens), hq, d, generator=g) - shift).to(torch.bfloat16).cuda()
    if fp8:
        # (code 0x80, torch's -0, is the format's NaN)
        k, v = (torch.where(t.abs() < 2.0 ** -6, 0.0, t).clamp(-200, 200)
                .to(torch.float8_e4m3fn).view(torch.uint8) for t in (k, v))
    else:
        k, v = k.to(torch.bfloat16), v.to(torch.bfloat16)
    k, v = k.cuda(), v.cuda()
    tables = torch.zeros(copies, max(blocks), dtype=torch.int32)
    o = 0
    for i, n in enumerate(blocks):
        tables[i, :n] = torch.arange(o, o + n)
        o += n
    cu = torch.tensor([0] + torch.tensor(q_lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    pl = torch.tensor(past, dtype=torch.int32)
    absent = torch.tensor([-1, nb, nb + 7, -5], dtype=torch.int32).expand(copies, 4)
    outs = [pa.prefill(q, k, v, t.cuda(), cu, p.cuda(), max(q_lens), scale=d ** -0.5)
            for t, p in ((tables, pl), (torch.cat([absent, tables], 1), pl + 64))]
    assert outs[0].float().abs().sum() > 0
    assert torch.equal(outs[0], outs[1])
