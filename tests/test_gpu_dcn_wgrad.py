"""The weight-gradient kernel (dcn_wgrad.hip) against float64: tile and part remainders, every
type, output rounding and non-finite operands.

Bound per sum: products exact (16-bit types) or to 2^-23 (fp32), fewer than M / 8 + 32 fp32
roundings of partial sums that stay below sum |a b|, and one rounding to the output type."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _reference(cols, dout, taps):
    m, k = cols.shape
    w = dout.double().t() @ cols.double()
    wa = dout.double().abs().t() @ cols.double().abs()
    c = k // taps
    to = [t.view(-1, taps, c).permute(0, 2, 1) for t in (w, wa)]
    return to[0], to[1]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16],
                         ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("m,c,cout,k", [(1, 8, 8, 3), (63, 16, 24, 3), (129, 40, 72, 3),
                                        (1025, 64, 136, 1), (5003, 96, 64, 3), (20000, 24, 200, 5)])
def test_weight_grad(dtype, m, c, cout, k):
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(m)
    cols = torch.randn(m, k * k * c, generator=g).to(dtype)
    dout = torch.randn(m, cout, generator=g).to(dtype)
    ref, ref_abs = _reference(cols, dout, k * k)
    for out_dtype in {dtype, torch.float32}:
        got = ext.dcn_weight_grad(cols.to(DEV), dout.to(DEV), k, k, out_dtype)
        assert got.dtype == out_dtype
        err = (got.double().cpu().reshape(ref.shape) - ref).abs()
        bound = (m / 8 + 34) * 2.0 ** -23 * ref_abs + EPS[out_dtype] * ref.abs() + 1e-7
        assert (err <= bound).all(), f"worst {(err / bound).max().item():.3f}"
    again = ext.dcn_weight_grad(cols.to(DEV), dout.to(DEV), k, k, out_dtype)
    assert torch.equal(got, again), "not the same on every run"


@pytest.mark.parametrize("v", [1 + 2.0 ** -7 - 2.0 ** -23, 1 + 2.0 ** -8 - 2.0 ** -17])
@pytest.mark.parametrize("m", [32, 64])
def test_weight_grad_equal_operands(m, v):
    """All products alike, so that the pieces left out add up: 2^-24 of the sum, and at most three
    fp32 roundings per 32 pixels."""
    import _modulated_deform_conv_ext as ext
    t = torch.full((m, 72), v, device=DEV)
    got = ext.dcn_weight_grad(t, t, 3, 3).double()
    ref = m * t[0, 0].double().item() ** 2
    assert (got - ref).abs().max().item() <= (3 * m / 32 + 1) * 2.0 ** -24 * ref


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["fp32", "bf16"])
def test_weight_grad_nonfinite(dtype):
    """Inf and NaN reach exactly the sums they reach in float64 (a zero times Inf is NaN, Inf
    times a value with no lower pieces is Inf)."""
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(3)
    m, c, cout = 700, 32, 48
    cols = torch.randint(-2, 3, (m, 9 * c), generator=g).to(dtype)
    dout = (torch.randint(0, 4, (m, cout), generator=g) + 0.5).to(dtype)
    cols[500, 40] = float("inf")
    dout[3, 7] = float("nan")
    dout[650, 20] = float("-inf")
    ref, _ = _reference(cols, dout, 9)
    got = ext.dcn_weight_grad(cols.to(DEV), dout.to(DEV), 3, 3, torch.float32)
    got = got.double().cpu().reshape(ref.shape)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    fin = torch.isfinite(ref)
    assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])
    assert torch.equal(got[fin], ref[fin]) and 0.9 < fin.double().mean() < 1  # small halves: exact


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16],
                         ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("b,c,h,w,kh,kw,pad,stride,dil", [
    (1, 8, 5, 6, 3, 3, 1, 1, 1), (2, 24, 17, 13, 3, 3, 1, 2, 1), (1, 72, 33, 47, 3, 3, 2, 1, 2),
    (3, 136, 9, 70, 1, 3, 0, 1, 1), (2, 264, 30, 3, 3, 3, 1, 1, 1)])
def test_split_backward_step(dtype, b, c, h, w, kh, kw, pad, stride, dil):
    """dcn_split_backward_nhwc against the column-to-image kernel plus the float64 gradients of
    the plain convolution: strides, dilations, rows shorter than a step's pixels, tiles that end
    inside a tap. The step's grad_y sums in fp32; 2e-6 of the sum of magnitudes covers its
    products and sums, then one rounding."""
    import _modulated_deform_conv_ext as ext
    import torch.nn.functional as F
    g = torch.Generator().manual_seed(c)
    t = kh * kw
    ho, wo = ((n + 2 * pad - dil * (k - 1) - 1) // stride + 1 for n, k in ((h, kh), (w, kw)))
    m = b * ho * wo
    x = torch.randn(b, h, w, c, generator=g).to(dtype).to(DEV)
    y = torch.randn(b, ho, wo, 3 * t, generator=g).to(dtype).to(DEV)
    dcol = torch.randn(m, t * c, generator=g).to(dtype).to(DEV)
    w_off = (0.2 * torch.randn(3 * t, c, kh, kw, generator=g)).to(dtype).to(DEV)
    sizes = (b, c, h, w, ho, wo, kh, kw, pad, pad, stride, stride, dil, dil)
    gx, gw, gb = ext.dcn_split_backward_nhwc(dcol, x, y, w_off, *sizes)
    s_x = torch.zeros(b, h, w, c, device=DEV)
    s_o, s_m = torch.empty(m, 2 * t, device=DEV), torch.empty(m, t, device=DEV)
    ext.modulated_deformable_col2im_nhwc_cuda(dcol, x, y, y, *sizes, 1, s_x, s_o, s_m)
    dy = torch.cat([s_o, s_m], 1).double().cpu().view(b, ho, wo, 3 * t).permute(0, 3, 1, 2)
    xs, ws = x.double().cpu().permute(0, 3, 1, 2), w_off.double().cpu()
    col = F.unfold(xs, (kh, kw), dil, pad, stride)

    def grads(wt, cols, d):
        flat = d.flatten(2)
        back = F.fold(wt.flatten(1).t() @ flat, (h, w), (kh, kw), dil, pad, stride)
        return (back.permute(0, 2, 3, 1), (flat @ cols.transpose(1, 2)).sum(0).view_as(wt),
                flat.sum((0, 2)))
    ref = grads(ws, col, dy)
    mag = grads(ws.abs(), col.abs(), dy.abs())
    add = (s_x.double().cpu(), 0.0, 0.0)
    for name, got, r, a, extra in zip(("grad_x", "grad_w_off", "grad_b_off"), (gx, gw, gb), ref, mag,
                                      add):
        assert got.dtype == dtype
        r = r + extra
        err = (got.double().cpu() - r).abs()
        # grad_x: the two column-to-image runs add their atomics in different orders
        bound = 2e-6 * (a + r.abs()) + EPS[dtype] * r.abs() + (1e-5 if name == "grad_x" else 1e-7)
        assert (err <= bound).all(), f"{name}: worst {(err / bound).max().item():.3f}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("rows,n", [(1, 8), (17, 64), (5000, 512), (333, 2056)])
def test_column_sums(dtype, rows, n):
    import _modulated_deform_conv_ext as ext
    g = torch.Generator().manual_seed(rows)
    a = torch.randn(rows, n, generator=g).to(dtype)
    got = ext.column_sums(a.to(DEV), torch.float32).double().cpu()
    bound = (rows + 64) * 2.0 ** -24 * a.double().abs().sum(0)
    assert ((got - a.double().sum(0)).abs() <= bound).all()
