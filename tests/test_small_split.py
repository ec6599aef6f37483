"""Workgroup width of the split-reduction kernel's spread form (host side of csrc/fused_sparse.hip):
32-channel workgroups where they add no round over 256 CUs."""
import pytest

from sparsesnn_amd import ops


@pytest.mark.parametrize("T,planes,rows,C_out,ch", [  # rows of 16 positions
    (4, 1, 1, 64, 32), (4, 1, 128, 64, 32), (4, 1, 129, 64, 64), (4, 2, 64, 128, 32), (4, 2, 65, 128, 64),
    (4, 2, 256, 64, 64), (4, 2, 300, 64, 64), (8, 1, 128, 64, 32), (8, 1, 129, 64, 64), (8, 1, 300, 64, 64),
    (8, 2, 128, 64, 32), (8, 2, 129, 64, 64), (8, 2, 256, 64, 64), (8, 2, 257, 64, 32), (8, 2, 384, 64, 32),
    (8, 2, 385, 64, 64), (1, 1, 128, 64, 32), (2, 2, 129, 64, 64),
])
def test_small_split(T, planes, rows, C_out, ch):
    spec = ops.ConvSpec(T=T, B=1, C_in=64, H=rows, W=16, C_out=C_out, weight_planes=planes)
    assert ops.fused_plan(spec).startswith("smallm<") and f",ch={ch}>" in ops.fused_plan(spec), ops.fused_plan(spec)
    soft = ops.ConvSpec(T=T, B=1, C_in=64, H=rows, W=16, C_out=C_out, weight_planes=planes, hard_reset=False)
    assert ",ch=64>" in ops.fused_plan(soft)  # the generic form has no narrow workgroups
