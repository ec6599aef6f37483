"""GPU parity of the LDS-staged kernel's epilogue instances (csrc/fused_sparse_lds.hip).

Calls without traces run the plain mode where no hard-reset one exists (soft reset, tau != 2, fp16
output) and with it two channel groups per wave on wide layers; traces keep the generic mode and one
group.  Each against the CPU oracle (oracle.reference_path: models/neurons.py LIF / IF over F.conv2d +
eval BN), ragged last tiles included.
"""
import pytest
import torch

from oracle import reference_path as ref
from sparsesnn_amd import ops
from tests.test_gpu_fused import run_case

pytestmark = pytest.mark.gpu


@pytest.fixture
def lds_route():
    ops.set_fused_kernel("lds")
    yield
    ops.set_fused_kernel("auto")


@pytest.mark.parametrize("T,planes,neuron,tau,v_reset,f16,state,traces,wide", [
    (8, 1, "if", 2.0, None, False, False, False, False),
    (8, 2, "lif", 1.5, 0.0, False, True, False, False),
    (4, 1, "lif", 3.0, 0.3, True, True, False, False),
    (4, 2, "lif", 2.0, 0.0, True, False, False, False),
    (2, 1, "if", 2.0, None, False, True, False, False),
    (1, 2, "lif", 2.0, None, False, False, False, False),
    (4, 1, "if", 2.0, None, False, False, False, True),
    (4, 2, "lif", 2.0, 0.0, False, False, False, True),
    (4, 2, "lif", 2.0, None, True, True, False, True),
    (4, 1, "lif", 1.5, 0.0, False, False, True, True),
])
def test_lds_epilogues(dev, lds_route, T, planes, neuron, tau, v_reset, f16, state, traces, wide):
    """wide: 65 x 63 pixels x 512 channels, enough waves for two channel groups each."""
    B, H, W, C_out = (1, 65, 63, 512) if wide else (2, 9, 11, 128)
    case = ref.make_layer_case(811 + T + planes, T=T, B=B, C_in=64, C_out=C_out, H=H, W=W, k=3, stride=1, padding=1,
                               fp16_weights=planes == 1, p_spike=0.3)
    out_enc = ops.ENC_F16 if f16 else ops.ENC_BITS
    spec = ops.ConvSpec(T=T, B=B, C_in=64, H=H, W=W, C_out=C_out, neuron=neuron, hard_reset=v_reset is not None,
                        tau=tau, v_threshold=0.5, v_reset=v_reset or 0.0, out_enc=out_enc, weight_planes=planes)
    plan = ops.fused_plan(spec, traces=traces, state=state)
    hard = v_reset is not None and tau == 2.0 and not f16
    assert plan.startswith("lds<") and plan.endswith(
        f"epi={'generic' if traces else 'lif_hard' if hard else 'plain'}>"), plan
    assert f"GPW={2 if wide and not traces else 1}," in plan, plan
    v0 = torch.rand((B, C_out, H, W), generator=torch.Generator().manual_seed(3)) * 0.4 if state else None
    rep, x_err, r, v_fin = run_case(dev, case, neuron=neuron, tau=tau, v_reset=v_reset, v_th=0.5, planes=planes,
                                    out_enc=out_enc, v0=v0, traces=traces)
    print(plan, rep, x_err)
    assert rep.ok, str(rep)
    assert x_err is None or x_err < 1e-4
    if state:  # spikes agree, so the membranes differ by the fp32 sums' rounding only
        assert torch.allclose(v_fin, r.v_final, rtol=1e-3, atol=1e-3)
    assert float(r.spikes.mean()) > 0.01
