"""The matrix-core stem at every block size: partial pixel blocks, images smaller than a block, one
and several steps beyond a group of four, both channel splits; spikes bit-identical to the neuron
run over the kernel's own fp32 output, which is checked against a float64 convolution."""
import pytest
import torch
import torch.nn.functional as F

from sparsesnn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [16, 12, 8])
@pytest.mark.parametrize("B,H,W,C_out,K,S,neuron,T,v_reset,tau", [
    (1, 5, 7, 64, 3, 1, "lif", 4, 0.0, 2.0),     # one partial block, four tiles per wave
    (2, 33, 45, 64, 7, 2, "lif", 8, 0.0, 2.0),   # two groups of four steps, ragged rows
    (3, 23, 130, 64, 3, 2, "lif", 1, None, 2.0),  # one step, soft reset, wide rows
    (2, 31, 31, 32, 3, 1, "if", 6, 0.25, 2.0),   # two tiles, nonzero reset value
    (1, 40, 24, 32, 7, 2, "lif", 5, 0.0, 1.5),   # general decay
    (2, 29, 45, 64, 7, 2, "lif", 8, None, 2.0),  # soft reset over full groups of four steps
    (1, 12, 19, 32, 3, 1, "if", 7, None, 2.0),   # and a rest of three
    (1, 16, 16, 64, 3, 1, "lif", 6, None, 3.0),  # soft reset, general decay, a rest of two
])
def test_stem_blocks(dev, env, nb, B, H, W, C_out, K, S, neuron, T, v_reset, tau):
    env("SENGINE_AMD_STEM_NB", nb)
    g = torch.Generator().manual_seed(H + K)
    x = torch.randn(B, 3, H, W, generator=g)
    w = torch.randn(C_out, 3, K, K, generator=g) * 2.0 / (3 * K * K) ** 0.5
    sc, bi = torch.rand(C_out, generator=g) + 0.5, torch.randn(C_out, generator=g) * 0.3
    spec = ops.ConvSpec(T=T, B=B, C_in=3, H=H, W=W, C_out=C_out, KH=K, KW=K, stride=S, padding=K // 2, neuron=neuron,
                        hard_reset=v_reset is not None, tau=tau, v_reset=v_reset or 0.0)
    hwio = w.permute(2, 3, 1, 0).contiguous().to(dev)
    # a 4-byte aligned output: the 16-byte stores may not assume more
    OH, OW = (H + 2 * (K // 2) - K) // S + 1, (W + 2 * (K // 2) - K) // S + 1
    out = torch.empty(B * OH * OW * C_out + 1, device=dev)[1:].view(B, OH, OW, C_out)
    out, spk = ops.stem_conv_bn_neuron(spec, x.to(dev), hwio, sc.to(dev), bi.to(dev), out=out)
    conv = lambda a, b: F.conv2d(a.double(), b.double(), None, S, K // 2).permute(0, 2, 3, 1) * sc.double()  # noqa: E731
    exact, mag = conv(x, w) + bi.double(), conv(x.abs(), w.abs())
    # n products and n - 1 sums in fp32, any order: (n + 1) eps of the absolute sum; 2 eps for the affine
    n, eps = 3 * K * K, 2.0 ** -24
    bound = (n + 1) * eps * mag + 2 * eps * (exact.abs() + mag + bi.abs().double())
    assert ((out.cpu().double() - exact).abs() <= bound).all()
    ref = ops.multistep_neuron_repeat(out.clone().view(-1), T, neuron, tau, 1.0, v_reset)
    assert torch.equal(spk.view(-1), ref.view(-1))
    _, only = ops.stem_conv_bn_neuron(spec, x.to(dev), hwio, sc.to(dev), bi.to(dev), want_out=False)
    assert torch.equal(only.view(-1), ref.view(-1))
