"""Which calls of the attention core are one kernel and which two (host side of csrc/ssa.hip)."""
import pytest

from sparsesnn_amd import ops


@pytest.mark.parametrize("T,B,N,C,heads,needs", [
    (4, 1, 196, 384, 8, False),    # measured 19.6 us as two kernels, 13.6 as one
    (4, 8, 196, 384, 8, False),    # 22.0 / 13.7
    (4, 11, 196, 384, 8, False),   # 25.7 / 13.7
    (4, 1, 784, 384, 8, True),     # 24.6 / 28.8
    (4, 8, 784, 384, 8, False),    # 38.9 / 29.1
    (4, 1, 3136, 384, 8, True),    # 59.2 / 86.1
    (4, 4, 3136, 384, 8, True),    # 72.0 / 86.9
    (4, 12, 3136, 384, 8, False),  # 102.7 / 89.4
    (8, 1, 64, 512, 8, False),     # 25.3 / 17.8
    (8, 1, 400, 512, 8, True),     # 28.8 / 46.9
    (8, 1, 576, 512, 8, True),     # 30.0 / 54.6
    (8, 11, 768, 512, 8, False),   # 106 / 70
    (1, 1, 3136, 256, 8, False),   # 39.8 / 18.5
])
def test_attention_route_follows_the_measurements(T, B, N, C, heads, needs):
    """One rule with and without a workspace (from eight pairs), on the faster side of measured shapes."""
    assert ops.attention_needs_kv(T, B, N, C, heads) == needs
    assert ops.attention_needs_kv(T, B, N, C, heads, workspace=True) == needs


def test_attention_route_below_eight_pairs():
    """An engine's launch list keeps its two launches there; a call without a workspace takes the one."""
    assert ops.attention_needs_kv(4, 2, 4, 128, 2, workspace=True) and not ops.attention_needs_kv(4, 2, 4, 128, 2)
