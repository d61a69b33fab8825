"""Which channels the two-states-a-lane scan (ops/csrc/mamba.hip scan_lanes_kernel) stages: eight threads a token read four channels each, in
one load where the rows allow it, also the threads of a last workgroup whose channels lie past the last one."""
import pytest

from vllm_distributed_amd.ops import native as N


@pytest.mark.parametrize("vec", [0, 1])
def test_staged_channels_lie_in_their_row(vec):
    first = N.lib().vda_scan_lane_channel
    for C in range(4, 300, 4) if vec else range(1, 300):
        for at in range(0, -(-C // 32) * 32, 4):
            c = first(at, C, vec)
            assert 0 <= c and c + (4 if vec else 1) <= C, (C, at, c)
            assert not vec or c % 4 == 0, (C, at, c)               # a load of four lies on its boundary
            assert at >= C or c == at, (C, at, c)                  # threads that have channels read their own
