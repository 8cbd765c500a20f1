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


# Rows, columns (SwiGLU: outputs) and K that reach every tiling, the two lowest
# with K steps of 128 (whole ones) and of 64; test_gemm_tiling.py holds the
# rule to these names.
TILINGS = {
    (152, 11, 320): "64x64", (183, 25, 512): "64x64",
    (213, 4434, 320): "64x128", (193, 4204, 384): "64x128",
    (593, 3327, 320): "128x128", (4177, 404, 320): "128x128",
    (1545, 4658, 384): "128x128 pair",
    (770, 4680, 320): "256x128", (3807, 1025, 320): "256x128",
    (1694, 4666, 320): "256x256", (2077, 3895, 320): "256x256",
}
TILINGS_SWIGLU = {
    (170, 128, 320): "64x64", (83, 256, 384): "64x64",
    (212, 2112, 320): "64x128", (243, 2112, 384): "64x128",
    (198, 4224, 320): "128x128",
    (409, 4160, 320): "128x128 pair",
    (642, 4864, 320): "256x128",
    (1191, 3328, 320): "256x256",
}


@pytest.mark.parametrize("m,n,k", list(TILINGS) + [
    (65, 8, 64), (65, 896, 4864), (127, 72, 192), (129, 100, 128), (257, 77, 64),
    (200, 520, 4096),
    (700, 1000, 896), (300, 2052, 896),  # N off the 16-byte stores
    (300, 2048, 960),
    (2000, 1024, 896),
    (6000, 900, 960),
    (4100, 4100, 512),
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
                                       (1500, 4864, 896), (3000, 704, 320)] +
                         list(TILINGS_SWIGLU))
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


@pytest.mark.parametrize("epi", ["bias", "add", "swiglu"])
def test_gemm_k_past_32_bit_offsets(pa, epi):
    """K of 2^23 and more takes the instance with 64-bit copy addresses."""
    m, n, k = 65, 128 if epi == "swiglu" else 9, 1 << 23
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.empty(m, k, dtype=torch.bfloat16, device="cuda"), torch.empty(
        n, k, dtype=torch.bfloat16, device="cuda")
    ref = torch.zeros(m, n, dtype=torch.float64, device="cuda")
    for c in range(0, k, 1 << 19):
        xc, wc = x[:, c:c + (1 << 19)], w[:, c:c + (1 << 19)]
        xc.copy_(torch.randn(xc.shape, generator=g, device="cuda"))
        wc.copy_(torch.randn(wc.shape, generator=g, device="cuda") * k ** -0.5)
        ref += xc.double() @ wc.double().t()
    # besides the roundings to bf16: 2^20 f32 additions, each off by at most
    # 2^-24 of a partial sum of at most about 5, independently: 2^10 2^-24 5
    f32 = 4 * 5 * 2.0 ** -14
    if epi == "swiglu":
        out = pa.linear(x, w, act=pa.ops.ACT_SILU_MUL)
        gate, up = ref[:, :64], ref[:, 64:]
        ref = torch.nn.functional.silu(gate) * up
        mag = ref.abs() + gate.abs() * up.abs()
        assert ((out.double() - ref).abs() <= 4 * RTOL * mag + 4 * f32).all()
        return
    b = torch.randn(m, n, generator=g, device="cuda").to(torch.bfloat16)
    if epi == "add":
        out, ref2 = pa.linear(x, w, out=b.clone(), add_to_out=True), ref + b.double()
    else:
        out, ref2 = pa.linear(x, w, b[0].contiguous()), ref + b[0].double()
    assert ((out.double() - ref2).abs() <= RTOL * (ref.abs() + ref2.abs()) + f32).all()
