"""Whether the keys of a prompt's tiles are cut into parts (vda_prefill_parts): sizes on either side of the line, by the measurements beside it."""
import pytest

from vllm_distributed_amd.ops import native as N


@pytest.mark.parametrize("new,prefix,Hq,Hkv,D,cut", [([1000], 0, 32, 8, 64, False), ([700], 0, 32, 8, 64, False), ([500] * 3, 0, 14, 2, 64, False),
                                                     ([300], 300, 32, 8, 128, True), ([100] * 4, 450, 32, 8, 128, False), ([100] * 4, 450, 16, 8, 256, True),
                                                     ([1000], 0, 8, 1, 128, True), ([100] * 2, 2000, 32, 8, 64, True), ([17], 1500, 64, 8, 128, True),
                                                     ([400], 0, 8, 1, 128, False), ([300] * 8, 2000, 32, 8, 128, False)])
def test_rule(new, prefix, Hq, Hkv, D, cut):
    assert (N.lib().vda_prefill_parts(len(new), sum(new), Hq, Hkv, D, max(new) + prefix) > 1) is cut
