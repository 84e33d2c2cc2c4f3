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
