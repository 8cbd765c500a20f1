"""The cache mirror's per-row block hashes and block-wise reads at the edges:
head dims off the 16 lanes of a row, tokens that overwrite slots of the same
call (more than 16 per block), reads past the ids that fit the kernel
arguments and of partial blocks."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
M64 = (1 << 64) - 1


def term(x):
    y = np.float32(abs(np.float32(x))) * np.float32(1000.0)
    if not y > 0:
        return 0
    return M64 if y >= 2.0 ** 64 else int(y)


def replay(rows, block, h, d, tokens):
    """{hash: block} after every token (rows: [T, H, D] values, tokens: (t, offset))."""
    state = np.zeros((h, 16, d), np.float32)
    out = {}
    for t, o in tokens:
        state[:, o] = rows[t]
        acc = 0
        for x in state.ravel():
            acc = (acc * 31 + term(x)) & M64
        out[acc] = block
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h,d", [(1, 2), (2, 16), (3, 24), (2, 64), (1, 130)])
def test_hashes_with_overwrites(pa, dtype, h, d):
    g = torch.Generator().manual_seed(h * d)
    # block 2: every slot, then slots again in another order (37 tokens); block 0: a few
    pos = list(range(16)) + [5, 5, 0, 15, 3] + list(range(15, -1, -1)) + [18, 17, 18, 30]
    t = len(pos)
    k = torch.randn(t, h, d, generator=g).to(dtype)
    k[3, 0, 0], k[7, 0, 1] = float("nan"), float("inf")
    v = torch.randn(t, h, d, generator=g).to(dtype)
    cache = pa.PagedKvCache(1, h, d, 4, dtype)
    cache.write_prefill_kv(0, [2, 0], pos, t, k.cuda(), v.cuda())
    rows = k.float().numpy()
    want = replay(rows, 2, h, d, [(i, p) for i, p in enumerate(pos) if p < 16])
    want.update(replay(rows, 0, h, d, [(i, p - 16) for i, p in enumerate(pos) if p >= 16]))
    assert cache.block_hashes(0) == want


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h,d,tokens", [(2, 64, 1), (2, 64, 255), (1, 128, 256 * 16), (1, 8, 257 * 16 - 3),
                                        (3, 24, 300), (1, 520, 33)])
def test_reads(pa, dtype, h, d, tokens):
    g = torch.Generator().manual_seed(tokens)
    blocks = (tokens + 15) // 16
    ids = torch.randperm(blocks + 3, generator=g)[:blocks].tolist()
    k, v = (torch.randn(tokens, h, d, generator=g).to(dtype).cuda() for _ in range(2))
    cache = pa.PagedKvCache(1, h, d, blocks + 3, dtype)
    cache.write_prefill_kv(0, ids, list(range(tokens)), tokens, k, v)
    rk, rv = cache.read_kv(0, ids, tokens)
    assert torch.equal(rk, k) and torch.equal(rv, v)
    short = max(1, tokens - 7)
    rk, rv = cache.read_kv(0, ids, short)
    assert torch.equal(rk, k[:short]) and torch.equal(rv, v[:short])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("blocks", [17, 256, 257])
def test_long_reads_return_complete(pa, dtype, blocks):
    """A read of more than 16 blocks returns after its stream has run it, so
    its rows can be used on any stream."""
    cache = pa.PagedKvCache(1, 1, 64, blocks, dtype)
    k = torch.randn(blocks * 16, 1, 64).to(dtype).cuda()
    cache.write_prefill_kv(0, list(range(blocks)), list(range(blocks * 16)), blocks * 16, k, -k)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        cache.read_kv(0, list(range(blocks)), blocks * 16)  # the outputs' memory is there
        torch.cuda._sleep(100_000_000)
        rk, rv = cache.read_kv(0, list(range(blocks)), blocks * 16)
        assert s.query()
    assert torch.equal(rk, k) and torch.equal(rv, -k)
