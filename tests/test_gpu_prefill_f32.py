"""f32 (and int8-in-f32) prefill on the matrix cores at the edges of its 16-token
tiles, 16-key blocks and key splits, against float64 attention."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(q, k, v, tables, q_lens, past, scale):
    hq, hkv = q.shape[1], k.shape[1]
    out, row = torch.zeros(q.shape, dtype=torch.float64), 0
    for n, p, ids in zip(q_lens, past, tables):
        ctx = p + n
        kk = k[ids].transpose(0, 1).reshape(hkv, -1, k.shape[3])[:, :ctx].double()
        vv = v[ids].permute(1, 0, 3, 2).reshape(hkv, -1, k.shape[3])[:, :ctx].double()
        for i in range(n):
            keys = p + i + 1  # each row over its own keys only
            for h in range(hq):
                g = h // (hq // hkv)
                w = torch.softmax(kk[g, :keys] @ q[row + i, h].double() * scale, 0)
                out[row + i, h] = w @ vv[g, :keys]
        row += n
    return out


def case(seed, hq, hkv, d, q_lens, past):
    g = torch.Generator().manual_seed(seed)
    blocks = [(a + b + 15) // 16 for a, b in zip(q_lens, past)]
    nb = sum(blocks) + 2
    perm = torch.randperm(nb, generator=g).tolist()
    tables, o = [], 0
    for n in blocks:
        tables.append(perm[o:o + n])
        o += n
    k = torch.randn(nb, hkv, 16, d, generator=g)
    v = torch.randn(nb, hkv, d, 16, generator=g)
    q = torch.randn(sum(q_lens), hq, d, generator=g)
    return q, k, v, tables


def run(pa, q, k, v, tables, q_lens, past, **kw):
    width = max(len(t) for t in tables)
    bt = torch.tensor([t + [-1] * (width - len(t)) for t in tables], dtype=torch.int32).cuda()
    cu = torch.tensor([0] + torch.tensor(q_lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    return pa.prefill(q.cuda(), k.cuda(), v.cuda(), bt, cu,
                      torch.tensor(past, dtype=torch.int32).cuda(), max(q_lens), **kw).cpu()


@pytest.mark.parametrize("hq,hkv,d", [(1, 1, 16), (4, 2, 32), (14, 2, 64), (3, 1, 64),
                                      (8, 2, 128), (5, 1, 256), (10, 2, 64)])
def test_against_float64(pa, hq, hkv, d):
    q_lens, past = [1, 17, 16, 33, 5], [0, 31, 64, 15, 130]
    q, k, v, tables = case(d + hq, hq, hkv, d, q_lens, past)
    for t, (a, b) in zip(tables, zip(q_lens, past)):
        n = (a + b) % 16
        if n:  # stale entries past the context
            k[t[-1], :, n:] = math.nan
            v[t[-1], :, :, n:] = math.inf
    out = run(pa, q, k, v, tables, q_lens, past)
    ref = reference(q, k, v, tables, q_lens, past, d ** -0.5)
    # f32 dot products of d terms (error about sqrt(d) 2^-24 |q| |k| scale in
    # the exponent, ~1e-6) and weighted sums of at most 147 keys
    assert (out.double() - ref).abs().max() <= 1e-5


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
def test_values_above_the_diagonal(pa, value):
    """A value or key that is not finite reaches the rows that attend it and no
    earlier one, within the same 16 x 32 step too."""
    q_lens, past = [40], [9]
    q, k, v, tables = case(5, 4, 2, 64, q_lens, past)
    at = 30  # key 30 = row 21
    v[tables[0][at // 16], :, 3, at % 16] = value
    out = run(pa, q, k, v, tables, q_lens, past)
    ref = reference(q, k, v, tables, q_lens, past, 0.125)
    assert torch.isfinite(out[:21]).all()
    assert torch.equal(torch.isfinite(out), torch.isfinite(ref))
    assert (out[:21].double() - ref[:21]).abs().max() <= 1e-5
    k2 = k.clone()
    v[tables[0][at // 16], :, 3, at % 16] = 0.5
    k2[tables[0][at // 16], :, at % 16, 7] = math.nan
    out = run(pa, q, k2, v, tables, q_lens, past)
    assert torch.isfinite(out[:21]).all() and torch.isnan(out[21:]).all()


@pytest.mark.parametrize("d", [64, 128])
def test_block_scales(pa, d):
    """int8-in-f32 caches: integer elements times the block's scale."""
    q_lens, past = [20, 3], [50, 0]
    q, k, v, tables = case(9, 6, 2, d, q_lens, past)
    k, v = (k * 40).round().clamp(-127, 127), (v * 40).round().clamp(-127, 127)
    scales = 0.01 + torch.rand(k.shape[0], generator=torch.Generator().manual_seed(1)) * 0.03
    out = run(pa, q, k, v, tables, q_lens, past, block_scales=scales.cuda())
    s = scales.double()[:, None, None, None]
    ref = reference(q, k.double() * s, v.double() * s, tables, q_lens, past, d ** -0.5)
    assert (out.double() - ref).abs().max() <= 2e-5


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("scale", [math.inf, -math.inf, math.nan])
def test_block_scale_above_the_diagonal(pa, d, scale):
    """A block's scale that is not finite (what a quantised write of an infinite
    value leaves) reaches the rows that attend the block and no earlier one,
    also where a 16-row tile straddles blocks; the scale of block 0 reaches no
    row through an id outside the pool."""
    q_lens, past = [40], [9]
    q, k, v, tables = case(11, 6, 2, d, q_lens, past)
    k, v = (k * 40).round().clamp(-127, 127), (v * 40).round().clamp(-127, 127)
    scales = torch.full((k.shape[0],), 0.02)
    s = scales.double()[:, None, None, None]
    ref = reference(q, k.double() * s, v.double() * s, tables, q_lens, past, d ** -0.5)
    bad = scales.clone()
    bad[tables[0][2]] = scale  # keys 32 .. 47: rows 23 .. 38
    out = run(pa, q, k, v, tables, q_lens, past, block_scales=bad.cuda())
    assert (out[:23].double() - ref[:23]).abs().max() <= 2e-5
    assert torch.isnan(out[23:]).all()
    # the pool's block 0 in no table, its scale not finite, one id outside the pool
    k, v = (torch.cat([torch.zeros_like(t[:1]), t]) for t in (k, v))
    tables = [[b + 1 for b in t] for t in tables]
    bad = torch.cat([torch.tensor([scale]), scales])
    tables[0][1] = -1  # keys 16 .. 31 absent
    out = run(pa, q, k, v, tables, q_lens, past, block_scales=bad.cuda())
    assert torch.isfinite(out).all()
    full = run(pa, q, k, v, tables, q_lens, past, block_scales=torch.cat([scales[:1], scales]).cuda())
    assert torch.equal(out, full)
