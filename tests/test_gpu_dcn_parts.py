"""16-bit fused forward with the reduction in parts (few pixels) against the float64 oracle with
columns rounded once to the type, and against the whole-K kernel (both round one fp32 sum of the
same products, so they differ by fp32 sums in another order and at most one rounding step)."""
import pytest
import torch

from _tol import check
from oracle import dcn as od

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (batch, cin, cout, h, w, relu) and the 16-row blocks of a workgroup that the shape takes on a
# 256-CU device: each height is a kernel of its own, and 4 and 5 keep other prefetch depths.
SHAPES = [(1, 128, 256, 3, 5, False, 2), (1, 512, 512, 29, 50, True, 3), (1, 256, 136, 17, 23, False, 2),
          (1, 320, 264, 9, 41, True, 2), (1, 512, 256, 58, 71, True, 4), (6, 512, 160, 15, 35, False, 4),
          (1, 1024, 512, 40, 40, False, 4), (3, 512, 160, 29, 50, True, 5), (1, 2048, 256, 50, 50, False, 5)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("b,cin,cout,h,w,relu,rows", SHAPES)
def test_fused_parts(dtype, b, cin, cout, h, w, relu, rows):
    import ctypes
    import _bevk
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(cin + h)
    sizes = (b, cin, h, w, h, w, cout, 3, 3, 1, 1, 1, 1, 1, 1)
    blocks = ctypes.c_int(-1)
    parts = _bevk.lib().bevk_dcn_nhwc_parts(_bevk._DTYPE_CODES[dtype], *sizes[:9], ctypes.addressof(blocks))
    assert parts > 1
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert blocks.value == rows
    x = torch.randn(b, h, w, cin, generator=g).to(dtype).to(DEV)
    off = (2.0 * torch.randn(b, h, w, 18, generator=g)).to(dtype).to(DEV)
    mask = torch.rand(b, h, w, 9, generator=g).to(dtype).to(DEV)
    weight = (0.05 * torch.randn(cout, cin, 3, 3, generator=g)).to(dtype).to(DEV)
    bias = torch.randn(cout, generator=g).to(dtype).to(DEV)
    out = ext.dcn_conv_nhwc(x, off, mask, weight, bias, *sizes)

    def oracle(o, m):
        return od.forward_nhwc(x.double().cpu(), o.double().cpu(), m.double().cpu(),
                               weight.double().cpu(), bias.double().cpu(), 1, 1, 1, col_dtype=dtype)
    check(out.cpu(), oracle(off, mask), dtype, "parts")
    whole = torch.empty_like(out)
    ext.dcn_fused_fwd_nhwc(x, off, mask, ext.dcn_pack_weight(weight), bias, *sizes, whole)
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    d = (out.double() - whole.double()).abs()
    assert (d <= ulp * whole.double().abs() + 1e-4).all()

    w_off = (0.02 * torch.randn(27, cin, 3, 3, generator=g)).to(dtype).to(DEV)
    b_off = torch.randn(27, generator=g).to(dtype).to(DEV)
    out, y = ext.dcn_layer_nhwc(x, w_off, b_off, weight, bias, *sizes, act_relu=relu)
    yref = od.offset_conv_nhwc(x.double().cpu(), w_off.double().cpu(), b_off.double().cpu(), 1, 1, 1)
    check(y.cpu(), yref, torch.float32, "y")
    ref = oracle(y[..., :18], torch.sigmoid(y[..., 18:].double()))
    check(out.cpu(), ref.clamp(min=0) if relu else ref, dtype, "layer in parts")


@pytest.mark.parametrize("b,c,cout,h,w,stride,dg", [
    (1, 32, 16, 1, 1, 1, 1), (2, 64, 72, 9, 7, 1, 1), (1, 64, 64, 32, 32, 1, 1),
    (3, 96, 160, 13, 10, 2, 1), (2, 64, 100, 11, 14, 1, 4), (1, 128, 264, 8, 9, 2, 2),
    (2, 256, 256, 20, 33, 1, 1)])
def test_layer_nchw_f32(b, c, cout, h, w, stride, dg):
    """The NCHW fp32 layer behind one call: planes of 4k, 2k and odd positions (the three widths of
    the NCHW stores), two K parts, deformable groups; against the float64 oracle."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(c + h)
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    x = torch.randn(b, c, h, w, generator=g)
    off = 2.0 * torch.randn(b, dg * 18, ho, wo, generator=g)
    mask = torch.rand(b, dg * 9, ho, wo, generator=g)
    weight = 0.1 * torch.randn(cout, c, 3, 3, generator=g)
    bias = torch.randn(cout, generator=g)
    out = ext.dcn_layer_nchw_f32(*(t.to(DEV) for t in (x, off, mask, weight, bias)), b, c, h, w, ho,
                                 wo, cout, 3, 3, 1, 1, stride, stride, 1, 1, dg)
    ref = od.forward_nchw(x.double(), off.double(), mask.double(), weight.double(), bias.double(),
                          (stride, stride), (1, 1), (1, 1), 1, dg)
    check(out.cpu(), ref, torch.float32, "nchw layer")


def test_small_layer_nonfinite_f32():
    """The small-problem kernel's plain fp32 path: NaN / Inf in the input and in the weight reach
    exactly the outputs they reach in float64."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(9)
    b, c, cout, h, w = 1, 64, 72, 12, 11
    x = torch.randn(b, c, h, w, generator=g)
    x[0, 7, 2, 3] = float("inf")
    x[0, 9, 8, 8] = float("nan")
    x[0, :, 5] = 0.0
    off, mask = torch.zeros(b, 18, h, w), torch.ones(b, 9, h, w)
    weight = 0.5 * torch.randint(1, 3, (cout, c, 3, 3), generator=g).float()
    weight[3, 5, 1, 1] = float("-inf")
    args = (b, c, h, w, h, w, cout, 3, 3, 1, 1, 1, 1, 1, 1, 1)
    out = ext.dcn_layer_nchw_f32(*(t.to(DEV) for t in (x, off, mask, weight)), None, *args)
    out = out.double().cpu()
    ref = od.forward_nchw(x.double(), off.double(), mask.double(), weight.double(), None, (1, 1),
                          (1, 1), (1, 1), 1, 1)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert inf.any() and torch.equal(out[inf], ref[inf])
    fin = torch.isfinite(ref)
    assert 0.5 < fin.double().mean() < 1
    check(out[fin], ref[fin], torch.float32, "finite outputs")
