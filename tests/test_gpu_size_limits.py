"""Behaviour at the 32-bit buffer-offset limit. The fast kernels address one batch of MSDA
value (one image of DCN input) through a buffer descriptor with a 32-bit range:
  * MSDA forward: a batch of value of 2 GiB or more takes msda_generic_kernel (64-bit
    indexing) and must still match the oracle, including samples past byte offset 2^31;
  * DCN fused NHWC forward: the whole input goes through one descriptor, so an input over
    2 GiB is rejected with an error before any launch (the reference's own NHWC gather
    stops earlier, at an int32 column element count, dcn_fused_nhwc_cuda.cu:37-40)."""
import pytest
import torch

from _tol import check
from oracle import msda as om

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def test_msda_forward_batch_over_2gib():
    """One level of 4100 x 4100 positions, one head of 32 fp32 channels: 2.15 GB of value
    per batch. Uniform samples put about half the corners past byte offset 2^31."""
    import msda_opt2
    H = W = 4100
    g = torch.Generator(device=DEV).manual_seed(51)
    value = torch.randn(1, H * W, 1, 32, generator=g, device=DEV)
    assert value.numel() * 4 >= 1 << 31
    nq, P = 64, 4
    gc = torch.Generator().manual_seed(52)
    loc = torch.rand(1, nq, 1, 1, P, 2, generator=gc)
    loc[0, 0, 0, 0, :, :] = torch.tensor([1.0 - 0.5 / W, 1.0 - 0.5 / H])  # near the last pixel
    attn = torch.softmax(torch.randn(1, nq, 1, P, generator=gc), -1).view(1, nq, 1, 1, P)
    shapes = torch.tensor([[H, W]], dtype=torch.int64)
    lsi = torch.tensor([0], dtype=torch.int64)
    out = msda_opt2.ms_deform_attn_forward(value, shapes.to(DEV), lsi.to(DEV), loc.to(DEV),
                                           attn.to(DEV))
    torch.cuda.synchronize()
    # fp32 sampling coordinates, as the kernels (one ulp of 4100 is 4.9e-4)
    ref = om.forward(value.cpu().double(), shapes, lsi, loc.double(), attn.double(),
                     coord_dtype=torch.float32)
    check(out.cpu(), ref, torch.float32, "msda batch over 2 GiB")


def test_dcn_input_over_2gib_rejected():
    """A 2100 x 2100 x 256 fp16 input (2.26 GB) through the fused NHWC forward: a clear
    error, no launch."""
    from modulated_deform_conv import fused_tl
    H = W = 2100
    C = Cout = 256
    x = torch.empty(1, H, W, C, dtype=torch.float16, device=DEV)
    off = torch.zeros(1, H, W, 18, dtype=torch.float16, device=DEV)
    mask = torch.ones(1, H, W, 9, dtype=torch.float16, device=DEV)
    weight = torch.zeros(Cout, C, 3, 3, dtype=torch.float16, device=DEV)
    with pytest.raises(RuntimeError, match="too large for 32-bit buffer offsets"):
        fused_tl.fused_dcn_forward_nhwc(x, off, mask, weight, None, 1, 1, 1)


def test_dcn_backward_on_a_map_past_the_layout_change():
    """The NCHW module's backward on a 2048 x 2048 map at stride 2, one position block more than
    the NHWC route's layout change takes. With zero offsets and a mask of ones the layer is the
    plain convolution: gradients of input, weight and bias against float64 (sums of 9, of 2^20
    and of 2^20 products; values near 1)."""
    import torch.nn.functional as F
    from modulated_deform_conv import ModulatedDeformConv2d
    g = torch.Generator().manual_seed(7)
    x = torch.randn(1, 4, 2048, 2048, generator=g)
    go = torch.randn(1, 2, 1024, 1024, generator=g)
    mod = ModulatedDeformConv2d(4, 2, 3, stride=2, padding=1).to(DEV)
    xd = x.to(DEV).requires_grad_()
    off = torch.zeros(1, 18, 1024, 1024, device=DEV, requires_grad=True)
    mask = torch.ones(1, 9, 1024, 1024, device=DEV)
    mod(xd, off, mask).backward(go.to(DEV))
    xr = x.double().requires_grad_()
    w = mod.weight.detach().cpu().double().requires_grad_()
    F.conv2d(xr, w, None, 2, 1).backward(go.double())
    check(xd.grad.cpu(), xr.grad, torch.float32, "grad_input")
    assert torch.isfinite(off.grad).all()
    # 2^20 products per sum: fp32 sums of magnitudes up to about 2^20
    for a, r in ((mod.weight.grad.cpu().double(), w.grad), (mod.bias.grad.cpu().double(),
                                                            go.double().sum((0, 2, 3)))):
        assert ((a - r).abs() <= 2.0 ** -24 * 2 ** 20).all()


def test_dcn_col2im_nhwc_on_a_map_of_9m_positions():
    """The per-sample column-to-image kernel past 2^23 output positions, where its float estimate of
    pair / taps is off by more than the one step it corrects. With zero offsets and a mask of ones
    a tap's gradient goes to one pixel: grad_x is the sum of 5 shifted columns, grad_mask a
    sum of 2 products (fp32)."""
    import _modulated_deform_conv_ext as ext
    import torch.nn.functional as F
    h = w = 3000
    c, t = 2, 5
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn(1, h, w, c, generator=g, device=DEV)
    dcol = torch.randn(h * w, t * c, generator=g, device=DEV)
    off, mask = torch.zeros(1, h, w, 2 * t, device=DEV), torch.ones(1, h, w, t, device=DEV)
    gx = torch.zeros_like(x)
    goff, gmask = torch.empty_like(off), torch.empty_like(mask)
    ext.modulated_deformable_col2im_nhwc_cuda(dcol, x, off, mask, 1, c, h, w, h, w, 1, t, 0, 2, 1, 1, 1,
                                              1, 1, gx, goff, gmask)
    d = dcol.view(h, w, t, c)
    wide = torch.zeros(h, w + 4, c, device=DEV)
    xp = F.pad(x[0], (0, 0, 2, 2))
    for k in range(t):
        wide[:, k:k + w] += d[:, :, k]
        assert torch.allclose(gmask[0, :, :, k], (d[:, :, k] * xp[:, k:k + w]).sum(-1), rtol=0, atol=1e-5)
    # values up to about 6: ten roundings of 2^-24 of sums below 32
    assert torch.allclose(gx[0], wide[:, 2:-2], rtol=0, atol=2e-5)
