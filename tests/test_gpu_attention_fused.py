"""The one-kernel attention core against exact integer attention: every head dim and T, token counts
around a 64-token group and a 16-token tile, products beyond 2048 (the high pieces), soft reset and a
general decay, and the K^T V copy for a caller's workspace."""
import numpy as np
import pytest
import torch

from oracle import packing as pk
from sparsesnn_amd import ops

pytestmark = pytest.mark.gpu


def _spikes(g, p, *shape):
    return torch.bernoulli(torch.full(shape, p), generator=g)


def _bits(x, dev):
    return torch.from_numpy(pk.pack_bits(x.reshape(-1, x.shape[-1]).numpy()).view(np.int32)).view(
        *x.shape[:-1], -1).to(dev)


@pytest.mark.parametrize("T,B,N,C,heads,p,neuron,tau,v_reset", [
    (4, 2, 196, 384, 8, 0.2, "lif", 2.0, 0.0),
    (4, 3, 1, 64, 4, 0.5, "lif", 2.0, 0.0),       # one token, head dim 16
    (1, 2, 63, 128, 4, 0.3, "lif", 2.0, 0.25),    # one step, a partial group
    (2, 1, 65, 96, 2, 0.3, "if", 2.0, 0.0),       # two groups
    (8, 2, 130, 256, 4, 0.3, "lif", 2.0, 0.0),    # eight steps of head dim 64
    (8, 1, 17, 96, 3, 0.4, "lif", 2.0, None),     # soft reset
    (4, 40, 33, 256, 8, 0.3, "lif", 3.0, 0.0),    # 320 pairs: two workgroups per CU; a general decay
    (4, 12, 2500, 128, 8, 0.95, "lif", 2.0, 0.0),  # 96 pairs of long grids; sums above 2048
    (4, 32, 790, 384, 12, 0.2, "lif", 2.0, 0.0),  # 384 pairs
])
def test_fused_attention_exact(dev, T, B, N, C, heads, p, neuron, tau, v_reset):
    assert not ops.attention_needs_kv(T, B, N, C, heads)
    g = torch.Generator().manual_seed(N + C)
    q, k, v = (_spikes(g, r, T * B, N, C) for r in (p, p, p))
    d = C // heads
    split = lambda t: t.view(T * B, N, heads, d).transpose(1, 2).contiguous()  # noqa: E731
    kv = split(k).transpose(-1, -2).contiguous() @ split(v)  # integers: exact in fp32
    x = (split(q) @ kv * 0.125).transpose(1, 2).reshape(T, B * N * C)
    mem, spk = torch.zeros(B * N * C), []
    for t in range(T):
        if neuron == "if":
            h = mem + x[t]
        else:
            h = mem * torch.tensor(1.0 - 1.0 / tau, dtype=torch.float32) + x[t] / tau
        s = h >= 0.5
        mem = torch.where(s, torch.full_like(h, v_reset) if v_reset is not None else h - 0.5, h)
        spk.append(s)
    ref = _bits(torch.stack(spk).float().view(T * B, N, C), "cpu")
    args = [_bits(t, dev) for t in (q, k, v)]
    kw = dict(neuron=neuron, tau=tau, v_threshold=0.5, v_reset=v_reset)
    out = ops.spiking_self_attention(*args, T, B, N, C, heads, **kw)
    assert torch.equal(out.cpu(), ref)
    ws = torch.full((T * B, heads, d, d), -1, dtype=torch.int32, device=dev)
    out = ops.spiking_self_attention(*args, T, B, N, C, heads, kv=ws, **kw)
    assert torch.equal(out.cpu(), ref) and torch.equal(ws.cpu(), kv.int())


def test_attention_refusals_of_the_one_kernel(dev):
    with pytest.raises(ops.SEngineError):  # what the two kernels refuse, the one refuses: scale not a power of two
        t = torch.zeros(4, 16, 2, dtype=torch.int32, device=dev)
        ops.spiking_self_attention(t, t, t, 4, 1, 16, 64, 4, scale=0.3)
