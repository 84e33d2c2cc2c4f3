"""The fp32 kernels on the bf16 matrix cores (dcn_f32.hip): tile heights, column widths, K
parts and remainders against float64, and non-finite operands.

Error bound: every product is exact to 2^-23 (pieces left out, both operands' cuts), the sum
of K terms is rounded fewer than K / 8 times in fp32, so |error| <= (K / 8 + 2) * 2^-23 *
sum_k |a_k w_k|."""
import pytest
import torch

from _tol import check
from oracle import dcn as od

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bounded(out, ref, ref_abs, k, what):
    err = (out.double().cpu() - ref).abs()
    bound = (k / 8 + 2) * 2.0 ** -23 * ref_abs + 1e-30
    assert (err <= bound).all(), f"{what}: worst err / bound {(err / bound).max().item():.3f}"


@pytest.mark.parametrize("m,k,c", [(1, 32, 16), (17, 64, 16), (144, 96, 32), (1000, 128, 16),
                                   (2333, 256, 48), (70, 32, 112)])
def test_gemm_f32(m, k, c):
    """Row blocks that end inside a tile, 1 and 2 columns tiles past a multiple of 64 / 128 /
    256, one and several K steps; values over 60 binades."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(m + k)
    a = torch.randn(m, k, generator=g) * 2.0 ** torch.randint(-30, 30, (m, k), generator=g)
    w = torch.randn(k, c, 3, 3, generator=g) * 0.1
    out = torch.full((m, 9 * c), float("nan"), device=DEV)
    ext.gemm_f32(a.to(DEV), ext.dcn_split_weight(w.to(DEV), True), 9 * c, out)
    wf = w.permute(0, 2, 3, 1).reshape(k, 9 * c).double()
    _bounded(out, a.double() @ wf, a.double().abs() @ wf.abs(), k, f"gemm {m}x{k}x{9 * c}")


# Operands whose pieces left out are large: cut off instead of rounded the first two leave 2^-21 of
# the product; rounded, the second leaves the most that can be, 2^-24.
EQUAL = [1 + 2.0 ** -7 - 2.0 ** -23, 1 + 2.0 ** -8 - 2.0 ** -17, 2 - 2.0 ** -23,
         -1 - 2.0 ** -7 + 2.0 ** -23]


@pytest.mark.parametrize("v", EQUAL)
@pytest.mark.parametrize("m,k", [(16, 32), (400, 32), (16, 64), (5000, 64)])
def test_gemm_equal_operands(m, k, v):
    """All products alike, so that what they leave out adds up: 2^-24 of the sum, and at most three
    fp32 roundings per 32 terms (two sums, one addition)."""
    import _modulated_deform_conv_ext as ext
    out = torch.empty(m, 144, device=DEV)
    w = torch.full((k, 16, 3, 3), v, device=DEV)
    ext.gemm_f32(torch.full((m, k), v, device=DEV), ext.dcn_split_weight(w, True), 144, out)
    ref = k * w[0, 0, 0, 0].double().item() ** 2
    assert (out.double() - ref).abs().max().item() <= (3 * k / 32 + 1) * 2.0 ** -24 * ref


@pytest.mark.parametrize("exp", [-90, -110])
def test_gemm_small_operands(exp):
    """Operands of 2^exp .. 2^(exp + 2) keep their 24 bits (the lowest of 2^-110 is bf16's smallest
    subnormal, 2^-133); the bound of every other product."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(-exp)
    m, k = 200, 256
    mant = (1 + 3 * torch.rand(m, k, generator=g)) * (torch.randint(0, 2, (m, k), generator=g) * 2 - 1)
    a = mant * 2.0 ** (exp // 2) * 2.0 ** (exp - exp // 2)
    w = torch.randn(k, 16, 3, 3, generator=g) * 2.0 ** 40
    out = torch.empty(m, 144, device=DEV)
    ext.gemm_f32(a.to(DEV), ext.dcn_split_weight(w.to(DEV), True), 144, out)
    wf = w.permute(0, 2, 3, 1).reshape(k, 144).double()
    scale = 2.0 ** (-exp - 40)  # the bound's 1e-30 is for results near 1
    _bounded(out.double() * scale, (a.double() @ wf) * scale, (a.double().abs() @ wf.abs()) * scale, k,
             f"2^{exp}")


def test_gemm_weight_near_the_largest_float():
    """A finite weight that rounds to Inf as a bf16: the tile runs in plain fp32 and keeps it."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(2)
    a = torch.randn(40, 64, generator=g) * 2.0 ** -100
    w = torch.randn(64, 16, 3, 3, generator=g)
    w[7, 3, 1, 1] = 3.4028234e38
    w[9, 4, 0, 2] = -3.3961776e38
    out = torch.empty(40, 144, device=DEV)
    ext.gemm_f32(a.to(DEV), ext.dcn_split_weight(w.to(DEV), True), 144, out)
    wf = w.permute(0, 2, 3, 1).reshape(64, 144).double()
    # 64 fused multiply-adds, each rounded once
    bound = 64 * 2.0 ** -24 * (a.double().abs() @ wf.abs()) + 1e-37
    assert ((out.double().cpu() - a.double() @ wf).abs() <= bound).all()


@pytest.mark.parametrize("b,cin,cout,h,w,stride", [
    (1, 32, 16, 5, 7, 1), (1, 64, 64, 32, 32, 1), (2, 32, 100, 23, 31, 2),
    (1, 96, 160, 20, 30, 1), (1, 64, 264, 41, 37, 1), (3, 32, 320, 60, 61, 1)])
@pytest.mark.parametrize("form", ["2T", "3T"])
def test_fused_forward_f32(b, cin, cout, h, w, stride, form):
    """Column tiles of 64, 128 and 256 (and past them), one and two K parts, both offset
    forms, against the float64 oracle at fp32 sampling positions."""
    from modulated_deform_conv import dcn_split_nhwc as ds
    g = torch.Generator().manual_seed(cin + cout)
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    x = torch.randn(b, h, w, cin, generator=g)
    y = 2.0 * torch.randn(b, ho, wo, 27, generator=g)
    weight = 0.1 * torch.randn(cout, cin, 3, 3, generator=g)
    bias = torch.randn(cout, generator=g)
    off, mask = y[..., :18].contiguous(), torch.sigmoid(y[..., 18:])
    args = (off, mask) if form == "2T" else (y, None)
    out = ds._fused_forward(x.to(DEV), *(t if t is None else t.to(DEV) for t in args),
                            weight.to(DEV), bias.to(DEV), stride, 1, 1)
    ref = od.forward_nhwc(x.double(), off.double(), mask.double(), weight.double(),
                          bias.double(), stride, 1, 1)
    check(out.cpu(), ref, torch.float32, f"fused f32 {form}")


def test_nonfinite_weight_f32():
    """NaN / Inf weights reach exactly the outputs they reach in float64, next to zeros in the
    input (0 * Inf) and to weights whose lower pieces are zero."""
    from modulated_deform_conv import fused_tl
    g = torch.Generator().manual_seed(5)
    x = torch.randn(1, 12, 13, 64, generator=g)
    x[0, 3:6] = 0.0
    off, mask = torch.zeros(1, 12, 13, 18), torch.ones(1, 12, 13, 9)
    weight = 0.5 * torch.randint(-2, 3, (80, 64, 3, 3), generator=g).float()
    weight[3, 5, 1, 1] = float("inf")
    weight[70, 60, 0, 2] = float("nan")
    weight[71, 1, 2, 2] = float("-inf")
    out = fused_tl.fused_dcn_forward_nhwc(x.to(DEV), off.to(DEV), mask.to(DEV), weight.to(DEV),
                                          None, 1, 1, 1).double().cpu()
    ref = od.forward_nhwc(x.double(), off.double(), mask.double(), weight.double(), None, 1, 1, 1)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isfinite(out), fin) and 0.5 < fin.double().mean() < 1
    check(out[fin], ref[fin], torch.float32, "finite outputs")
