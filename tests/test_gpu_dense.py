"""The dense fallback conv at the edges of its tiles and stages, against a float64 convolution."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import packing as pk
from sparsesnn_amd import ops

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24  # fp32 unit roundoff


@pytest.mark.parametrize("T,B,C,H,W,C_out,k,stride,pad,dil", [
    (4, 1, 32, 5, 3, 64, 3, 1, 1, 1),       # one k-step per stage, rows of one partial tile
    (1, 1, 64, 1, 1, 64, 1, 1, 0, 1),       # a single row, a single stage
    (4, 2, 96, 9, 7, 128, 5, 2, 2, 1),      # odd channel count, strided window
    (8, 3, 128, 11, 6, 64, 3, 1, 2, 2),     # four k-steps per stage, dilation
    (2, 1, 192, 8, 8, 192, 3, 1, 0, 1),     # two k-steps per stage, no padding
    (1, 1, 32, 12, 12, 64, 9, 1, 4, 1),     # more than 64 taps
    (4, 16, 64, 41, 39, 64, 1, 1, 0, 1),    # 1,600 units: two row tiles per wave, ragged last tile
    (4, 10, 256, 25, 25, 256, 3, 1, 1, 1),  # 1,564 units over several output groups
    (4, 4, 32, 52, 59, 64, 3, 1, 1, 1),     # 767 units: the last with one row tile per wave
    (4, 4, 96, 55, 56, 64, 3, 1, 1, 1),     # 770: two
])
@pytest.mark.parametrize("in_enc,planes", [(ops.ENC_BITS, 1), (ops.ENC_F16, 1), (ops.ENC_BITS, 2), (ops.ENC_F16, 2)])
def test_dense_conv_edges(dev, T, B, C, H, W, C_out, k, stride, pad, dil, in_enc, planes):
    g = torch.Generator().manual_seed(C + k)
    x = torch.bernoulli(torch.full((T * B, C, H, W), 0.3), generator=g)
    w = torch.randn((C_out, C, k, k), generator=g) * (2 / (k * k * C)) ** 0.5
    if planes == 1:
        w = w.half().float()
    scale, bias = torch.rand(C_out, generator=g) + 0.5, torch.randn(C_out, generator=g)
    spec = ops.ConvSpec(T=T, B=B, C_in=C, H=H, W=W, C_out=C_out, KH=k, KW=k, stride=stride, padding=pad, dilation=dil,
                        in_enc=in_enc, weight_planes=planes)
    nhwc = x.permute(0, 2, 3, 1).contiguous()
    data = torch.from_numpy(pk.pack_bits(nhwc.reshape(-1, C).numpy()).view(np.int32)) if in_enc == ops.ENC_BITS \
        else nhwc.half()
    y = ops.dense_conv_bn(spec, data.to(dev), ops.pack_dense_weights(spec, w.to(dev)), scale.to(dev), bias.to(dev))
    conv = lambda ww: F.conv2d(x.double(), ww.double(), None, stride, pad, dil).permute(0, 2, 3, 1)  # noqa: E731
    s64 = scale.double()
    exact, mag = conv(w) * s64 + bias.double(), conv(w.abs()) * s64
    # a sum of n fp32 products in any order is within n eps of its absolute sum (spikes are exact
    # and so are fp16 weights times them; two fp16 planes hold a weight to 2^-22); the affine adds 2 eps
    n = k * k * C * planes
    bound = (n * EPS + (2.0 ** -21 if planes == 2 else 0.0)) * mag + 2 * EPS * (exact.abs() + mag + bias.abs().double())
    assert ((y.cpu().double() - exact).abs() <= bound).all()
