"""The tiled RoPE + KV-cache write against the one-token kernel it stands in
for (which still takes rows that are not 16-byte aligned, and fewer than 512
tokens of at most 512 rotation pairs): equal bit for bit, for token counts
around the 16-token tiles, runs of slots at every block offset, scattered and
skipped slots, and every head dim it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def slots_of(kind, t, nb, g):
    if kind == "scattered":
        s = torch.randperm(nb * 16, generator=g)[:t]
        s[::7] = -1
        return s
    start = int(kind)  # a prompt's consecutive slots from an offset, over shuffled blocks
    perm = torch.randperm(nb, generator=g)
    pos = torch.arange(start, start + t)
    return perm[pos // 16] * 16 + pos % 16


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (32, 8, 128), (4, 4, 16), (3, 1, 256), (6, 2, 80),
                                      (16, 2, 64), (48, 24, 16), (5, 1, 256), (12, 2, 80)])
@pytest.mark.parametrize("t,kind", [(1, "scattered"), (15, "3"), (16, "0"), (17, "15"), (40, "scattered"),
                                    (100, "9"), (333, "0"), (511, "3"), (512, "scattered"),
                                    (600, "7")])
def test_equals_one_token_kernel(pa, dtype, hq, hkv, d, t, kind):
    g = torch.Generator().manual_seed(t + d)
    nb = (t + 47) // 16 + 2
    row = (hq + 2 * hkv) * d
    data = torch.randn(t, row, generator=g).to(dtype)
    slots = slots_of(kind, t, nb, g).to(torch.int64).cuda()
    pos = torch.randint(0, 40000, (t,), generator=g).cuda()
    inv = torch.from_numpy(pa.rope_inv_freq(d, 1e6)).cuda()
    results = []
    for shift in (0, 1):  # 1: rows off 16-byte alignment, the one-token kernel
        flat = torch.zeros(t * row + shift, dtype=dtype, device="cuda")
        qkv = flat[shift:].view(t, hq + 2 * hkv, d)
        qkv.copy_(data.view(t, hq + 2 * hkv, d))
        kc, vc = pa.ops.new_cache(nb, hkv, d, dtype)
        kc.fill_(3.0)
        vc.fill_(5.0)
        pa.rope_reshape_and_cache(qkv[:, :hq], qkv[:, hq:hq + hkv], qkv[:, hq + hkv:], kc, vc,
                                  slots, pos, inv)
        results.append((qkv.clone(), kc, vc))
    for a, b in zip(*results):
        assert torch.equal(a, b)
