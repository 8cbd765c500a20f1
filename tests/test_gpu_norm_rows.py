"""pa_rms_norm / pa_layer_norm around the widths where the row kernel changes
(a wavefront or a workgroup per row, the widest row, widths and addresses off
16 bytes) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype,hidden", [
    (torch.bfloat16, h) for h in (8, 512, 2040, 2048, 2056, 4096, 8192, 8200, 36)
] + [(torch.float32, h) for h in (4, 260, 1024, 1028, 4096, 4100, 18)])
@pytest.mark.parametrize("rows,layer,shift", [(1, False, 0), (5, True, 0), (6, False, 1),
                                              (3, True, 1)])
def test_norms(pa, dtype, hidden, rows, layer, shift):
    g = torch.Generator().manual_seed(hidden + rows)

    def make(*shape, scale=1.0, mean=0.0):
        n = 1
        for d in shape:
            n *= d
        flat = torch.zeros(n + shift, dtype=dtype, device=DEV)  # `shift` elements off 16 bytes
        flat[shift:] = (torch.randn(n, generator=g) * scale + mean).to(dtype).cuda()
        return flat[shift:].view(*shape)

    x, a = make(rows, hidden, scale=2.0, mean=0.5), make(rows, hidden)
    w, b = make(hidden, scale=0.1, mean=1.0), make(hidden, scale=0.1)
    s = (x.float() + a.float()).to(dtype)
    z = s.double()
    if layer:
        z = z - z.mean(-1, keepdim=True)
    ref = z / torch.sqrt(z.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()
    if layer:
        ref = ref + b.double()
        out = pa.layer_norm(x, w, 1e-6, bias=b, add=a)
    else:
        out = pa.rms_norm(x, w, 1e-6, add=a)
    assert torch.equal(x, s)  # the residual, in the storage type
    # one rounding of the result (2^-9 relative in bf16), and f32 sums of at most
    # 4 x 8 products a lane and 8 levels of a tree: 48 roundings of 2^-24, of
    # which the root halves the relative part; the centred value's absolute error
    # is that of the mean, magnified by 1 / deviation < 4 and the weight < 2
    tol = 48 * 2.0 ** -24 * 8
    rel = tol + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)
    torch.testing.assert_close(out.double(), ref, atol=tol, rtol=rel)
