"""The tiled GEMM behind pa_linear at the edges of its tilings: rows around
the tile heights, output widths off the tiles and off the 16- and 8-byte
stores, K steps of 64 and 128 and K shorter than the copy pipeline, every
epilogue, against float64 of the same bf16 operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# One bf16 rounding of an f32 sum: half an ulp, 2^-9 of the value, plus the
# f32 sum's own error (K products of |x w| summed in f32: below 2^-14 of
# the sum of magnitudes at these K), SwiGLU and the residual one rounding more.
RTOL = 2.0 ** -8


def bound(ref, mag, roundings):
    return roundings * RTOL * ref.abs() + mag * 2.0 ** -14 + 1e-6


@pytest.mark.parametrize("m,n,k", [
    (65, 8, 64), (65, 896, 4864), (127, 72, 192), (129, 100, 128), (257, 77, 64),
    (200, 520, 4096),          # 64 x 64
    (700, 1000, 896), (300, 2052, 896),  # 64 x 128, N off the 16-byte stores
    (300, 2048, 960),          # 64 x 128, K steps of 64
    (2000, 1024, 896),         # 128 x 128 with K groups
    (6000, 900, 960),          # two workgroups per CU, or 256 x 128
    (4100, 4100, 512),         # 256 x 256
])
@pytest.mark.parametrize("epi", ["none", "bias", "add"])
def test_gemm_edges(pa, m, n, k, epi):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(torch.bfloat16)
    ref = x.double() @ w.double().t()
    mag = (x.double().abs() @ w.double().abs().t())
    if epi == "bias":
        # a view at an odd offset: the bias has no alignment of its own
        b = torch.randn(n + 1, generator=g, device="cuda").to(torch.bfloat16)[1:]
        out = pa.linear(x, w, b)
        ref, roundings = ref + b.double(), 1
    elif epi == "add":
        res = torch.randn(m, n, generator=g, device="cuda").to(torch.bfloat16)
        out = pa.linear(x, w, out=res.clone(), add_to_out=True)
        err = (out.double() - (ref + res.double())).abs()
        assert (err <= RTOL * (ref + res.double()).abs() + bound(ref, mag, 1)).all()
        return
    else:
        out, roundings = pa.linear(x, w), 1
    assert ((out.double() - ref).abs() <= bound(ref, mag, roundings)).all()


@pytest.mark.parametrize("m,inter,k", [(65, 64, 64), (333, 4864, 896), (129, 192, 128),
                                       (1500, 4864, 896), (3000, 704, 320)])
def test_gemm_swiglu_edges(pa, m, inter, k):
    g = torch.Generator(device="cuda").manual_seed(m + inter + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * inter, k, generator=g, device="cuda") * k ** -0.5).to(torch.bfloat16)
    out = pa.linear(x, w, act=pa.ops.ACT_SILU_MUL)
    y = x.double() @ w.double().t()
    gate, up = y[:, :inter], y[:, inter:]
    ref = torch.nn.functional.silu(gate) * up
    # gate and up are rounded to bf16 first: |d silu / d gate| <= 1.1
    err = (out.double() - ref).abs()
    assert (err <= 4 * RTOL * (ref.abs() + gate.abs() * up.abs()) + 1e-3).all()


def test_gemm_rows_past_m_untouched(pa):
    """Outputs past the last row and column stay as they were."""
    m, n, k = 130, 200, 128
    x = torch.randn(m, k, device="cuda").to(torch.bfloat16)
    w = torch.randn(n, k, device="cuda").to(torch.bfloat16)
    buf = torch.full((m + 64, n), 7.0, dtype=torch.bfloat16, device="cuda")
    pa.linear(x, w, out=buf[:m])
    assert (buf[m:] == 7.0).all()
