"""Vector and scalar forms of the streaming kernels (neuron, spike packing, spike max-pool): every
form at the sizes and alignments that select it, against the oracle or plain torch."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import packing as pk
from sparsesnn_amd import ops

pytestmark = pytest.mark.gpu


def _shifted(t, off):
    """t's values at `off` elements past an allocation's start (off 0: 16-byte aligned)."""
    buf = torch.empty(t.numel() + off, dtype=t.dtype, device=t.device)
    buf[off:] = t.flatten()
    return buf[off:].view(t.shape)


@pytest.mark.parametrize("neuron,tau,v_reset", [("lif", 2.0, 0.0), ("lif", 3.0, 0.25), ("if", 2.0, None),
                                                ("lif", 2.0, None)])
@pytest.mark.parametrize("T,n,off,enc", [(1, 32, 0, ops.ENC_BITS), (3, 1056, 0, ops.ENC_BITS),
                                         (4, 64 * 37, 0, ops.ENC_BITS), (4, 64 * 37, 1, ops.ENC_BITS),
                                         (9, 4096, 0, ops.ENC_BITS), (4, 1028, 0, ops.ENC_F16),
                                         (5, 1030, 0, ops.ENC_F16), (4, 1028, 2, ops.ENC_F16),
                                         # four elements per thread: more than the chip's 524,288 threads
                                         (4, 524288, 0, ops.ENC_BITS), (1, 524320, 0, ops.ENC_BITS),
                                         (6, 524320, 0, ops.ENC_BITS), (4, 524320, 1, ops.ENC_BITS),
                                         (3, 524292, 0, ops.ENC_F16), (5, 524294, 0, ops.ENC_F16),
                                         (4, 524292, 2, ops.ENC_F16)])
def test_neuron_forms(dev, neuron, tau, v_reset, T, n, off, enc):
    g = torch.Generator().manual_seed(T * n + off)
    x = torch.randn((T, n), generator=g) * 1.5 + 0.5
    v0 = torch.rand(n, generator=g) - 0.3
    v, spikes, hs = v0.clone(), [], []
    for t in range(T):
        if neuron == "lif":
            dec = torch.tensor(1.0 - 1.0 / tau, dtype=torch.float32)
            h = v * dec + x[t] / tau
        else:
            h = v + x[t]
        s = h >= 1.0
        v = torch.where(s, torch.full_like(h, v_reset) if v_reset is not None else h - 1.0, h)
        spikes.append(s)
        hs.append(h)
    state, trace = _shifted(v0.to(dev), off), _shifted(torch.zeros(T, n, device=dev), off)
    out = ops.multistep_neuron(_shifted(x.to(dev), off), T, neuron, tau, 1.0, v_reset, state=state, out_enc=enc,
                               h_trace=trace)
    got = (pk.unpack_bits(out.cpu().numpy().view(np.uint32).reshape(-1, 1), 32).reshape(T, n) if enc == ops.ENC_BITS
           else out.view(T, n).float().cpu().numpy())
    # the same fp32 operations in the same order: equal bit for bit
    assert np.array_equal(got, torch.stack(spikes).float().numpy())
    assert torch.equal(trace.cpu(), torch.stack(hs))
    assert torch.equal(state.cpu(), v)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("off", [0, 1, 4])
@pytest.mark.parametrize("n_pos,C", [(1, 32), (7, 96), (301, 64)])
def test_pack_unpack_alignment(dev, dtype, off, n_pos, C):
    g = torch.Generator().manual_seed(n_pos + C)
    x = torch.randn((n_pos, C), generator=g).to(dtype)
    x[torch.rand((n_pos, C), generator=g) < 0.5] = 0
    tiny = 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -149  # the smallest subnormals are spikes, -0 is none
    x.view(-1)[:6] = torch.tensor([tiny, -tiny, -0.0, float("nan"), float("-inf"), 1.0], dtype=dtype)
    bits = ops.pack_spikes(_shifted(x.to(dev), off))
    on = (x.float() != 0) if dtype == torch.float16 else x.ne(0)
    assert np.array_equal(bits.cpu().numpy().view(np.uint32), pk.pack_bits(on.float().numpy()))
    back = ops.unpack_spikes(bits, C, dtype, out=_shifted(torch.empty(n_pos, C, dtype=dtype, device=dev), off))
    assert torch.equal(back.cpu(), on.to(dtype))


@pytest.mark.parametrize("C", [32, 64, 96, 128, 384])
@pytest.mark.parametrize("H,W,k,stride,pad", [(1, 1, 3, 2, 1), (7, 10, 3, 2, 1), (8, 5, 2, 2, 0), (9, 9, 2, 1, 1),
                                              (6, 7, 5, 3, 2), (5, 5, 3, 1, 0), (4, 4, 1, 2, 0)])
@pytest.mark.parametrize("off", [0, 1])
def test_maxpool_forms(dev, C, H, W, k, stride, pad, off):
    g = torch.Generator().manual_seed(C + H)
    x = torch.bernoulli(torch.full((3, H, W, C), 0.2), generator=g)
    bits = torch.from_numpy(pk.pack_bits(x.reshape(-1, C).numpy()).view(np.int32)).to(dev)
    exp = F.max_pool2d(x.permute(0, 3, 1, 2), k, stride, pad).permute(0, 2, 3, 1).contiguous()
    out = ops.maxpool_spikes(_shifted(bits, off), 3, H, W, C, k, stride, pad)
    assert np.array_equal(out.cpu().numpy().view(np.uint32).reshape(-1, C // 32),
                          pk.pack_bits(exp.reshape(-1, C).numpy()))
