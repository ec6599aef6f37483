"""The split-reduction kernel's spread epilogue against an exact evaluation: weights, BN and decay are
chosen so that every product, sum and membrane is exact in fp32, so spikes and membranes must be
equal whatever the order of the sums."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import packing as pk
from sparsesnn_amd import ops, sparsity

pytestmark = pytest.mark.gpu


def _case(T, B, C, H, W, C_out, k, stride, seed, density=0.3):
    g = torch.Generator().manual_seed(seed)
    x = torch.bernoulli(torch.full((T * B, H, W, C), density), generator=g)
    w = torch.randint(-32, 33, (C_out, C, k, k), generator=g).float() / 64  # 2^-6 steps
    w = sparsity.prune_conv_2_4(w)
    scale = 2.0 ** torch.randint(-1, 2, (C_out,), generator=g).float()
    bias = torch.randint(-16, 33, (C_out,), generator=g).float() / 32
    y = F.conv2d(x.permute(0, 3, 1, 2).double(), w.double(), None, stride, k // 2).permute(0, 2, 3, 1)
    return x, w, scale, bias, y * scale.double() + bias.double()


def _neuron(y, T, neuron, v0):
    y = y.view(T, -1, *y.shape[1:])
    v, s = v0.double(), []
    for t in range(T):
        v = v * 0.5 + y[t] * 0.5 if neuron == "lif" else v + y[t]
        s.append(v >= 1.0)
        v = torch.where(s[-1], torch.zeros_like(v), v)
    return torch.cat(s), v


def _bits(x):
    return torch.from_numpy(pk.pack_bits(x.reshape(-1, x.shape[-1]).float().numpy()).view(np.int32))


SHAPES = [  # T, B, C, H, W, C_out, k, stride
    (4, 1, 64, 9, 7, 64, 3, 1),       # a ragged last position tile, 32-channel workgroups
    (4, 8, 64, 16, 16, 64, 3, 1),     # 128 workgroups of 64 channels: the last that run as pairs
    (4, 1, 64, 43, 48, 64, 3, 1),     # 129: 64-channel workgroups
    (4, 7, 64, 25, 23, 64, 3, 1),     # 252 and 256: the last of one round
    (4, 16, 64, 16, 16, 64, 3, 1),
    (1, 2, 64, 5, 5, 128, 1, 1),      # one chunk for eight waves
    (2, 1, 320, 6, 6, 64, 3, 2),      # 45 chunks
    (8, 2, 128, 11, 9, 192, 3, 2),    # two rounds of timesteps
    (8, 9, 64, 22, 22, 64, 1, 1),     # the same, 273 workgroups: pairs with two planes, whole with one
    (8, 13, 64, 22, 22, 64, 1, 1),    # 394: whole
    (4, 3, 128, 2, 2, 64, 3, 1),      # flat layout (four output pixels)
    (4, 5, 64, 3, 3, 128, 5, 1),      # 5x5 window, mostly padding
]


@pytest.mark.parametrize("planes", [1, 2])
@pytest.mark.parametrize("neuron,state", [("lif", False), ("if", True), ("lif", True)])
@pytest.mark.parametrize("T,B,C,H,W,C_out,k,stride", SHAPES)
def test_spread_epilogue_exact(dev, T, B, C, H, W, C_out, k, stride, neuron, state, planes):
    x, w, scale, bias, y = _case(T, B, C, H, W, C_out, k, stride, C + H)
    spec = ops.ConvSpec(T=T, B=B, C_in=C, H=H, W=W, C_out=C_out, KH=k, KW=k, stride=stride, padding=k // 2,
                        neuron=neuron, weight_planes=planes)
    assert ops.fused_plan(spec, state=state).startswith("smallm<")
    v0 = torch.randint(-8, 9, y.shape[1:], generator=torch.Generator().manual_seed(1)).float() / 8
    v0 = v0.expand(B, *v0.shape).contiguous() if state else torch.zeros(B, *y.shape[1:])
    s_ref, v_ref = _neuron(y, T, neuron, v0)
    mem = v0.reshape(-1, C_out).to(dev) if state else None
    values, meta, _ = ops.compress_2_4(spec, w.to(dev))
    out = ops.fused_sparse_conv_bn_lif(spec, _bits(x).to(dev), values, meta, scale.to(dev), bias.to(dev), state=mem)
    assert torch.equal(out.cpu().view(-1), _bits(s_ref).view(-1))
    if state:
        assert torch.equal(mem.cpu().double(), v_ref.reshape(-1, C_out))


@pytest.mark.parametrize("res_planes,out_planes", [(1, 2), (2, 2), (3, 5)])
@pytest.mark.parametrize("T,B,C,H,W,C_out,k,stride", [SHAPES[0], SHAPES[4], SHAPES[7], SHAPES[10]])
def test_spread_residual_planes_exact(dev, T, B, C, H, W, C_out, k, stride, res_planes, out_planes):
    x, w, scale, bias, y = _case(T, B, C, H, W, C_out, k, stride, C + H)
    spec = ops.ConvSpec(T=T, B=B, C_in=C, H=H, W=W, C_out=C_out, KH=k, KW=k, stride=stride, padding=k // 2)
    s_ref, _ = _neuron(y, T, "lif", torch.zeros(B, *y.shape[1:]))
    # residual values that leave room for the spike in out_planes bits
    top = min((1 << res_planes) - 1, (1 << out_planes) - 2)
    r = torch.randint(0, top + 1, s_ref.shape, generator=torch.Generator().manual_seed(3))
    planes_of = lambda a, n: torch.cat([(a >> p) & 1 for p in range(n)], dim=-1)  # noqa: E731
    values, meta, _ = ops.compress_2_4(spec, w.to(dev))
    out = ops.fused_sparse_conv_bn_lif_add(spec, _bits(x).to(dev), values, meta, scale.to(dev), bias.to(dev),
                                           _bits(planes_of(r, res_planes)).to(dev), res_planes, out_planes)
    assert torch.equal(out.cpu().view(-1), _bits(planes_of(r + s_ref.long(), out_planes)).view(-1))


def test_spread_pair_and_split_exact(dev):
    """A conv and its downsample in one launch, and channel-split output planes."""
    T, B, C, H, W = 4, 3, 64, 10, 10
    x, w0, sc0, bi0, y0 = _case(T, B, C, H, W, 128, 3, 2, 5)
    x1, w1, sc1, bi1, y1 = _case(T, B, C, H, W, 128, 1, 2, 5)
    assert torch.equal(x, x1)
    specs = [ops.ConvSpec(T=T, B=B, C_in=C, H=H, W=W, C_out=128, KH=k, KW=k, stride=2, padding=k // 2) for k in (3, 1)]
    blobs = [ops.compress_2_4(s, w.to(dev))[:2] for s, w in zip(specs, (w0, w1))]
    bn = [t.to(dev) for t in (sc0, bi0, sc1, bi1)]
    data = _bits(x).to(dev)
    o0, o1 = ops.fused_sparse_conv_bn_lif_pair(*specs, data, *blobs[0], *bn[:2], *blobs[1], *bn[2:])
    zero = torch.zeros(B, *y0.shape[1:])
    refs = [_neuron(y, T, "lif", zero)[0] for y in (y0, y1)]
    for o, r in zip((o0, o1), refs):
        assert torch.equal(o.cpu().view(-1), _bits(r).view(-1))
    sp = ops.fused_sparse_conv_bn_lif_split(specs[0], data, *blobs[0], *bn[:2], 64).cpu()
    for i in range(2):
        assert torch.equal(sp[i].view(-1), _bits(refs[0][..., 64 * i:64 * i + 64]).view(-1))
