"""Which 16-bit expert layers take 256-row tiles (ops._moe_wide_pays): where single experts past a tile's rows open another round over
the CUs, they do not.  Layers by experts, hidden and intermediate width, and rows an expert; times in the rule's comment."""
import pytest

from vllm_distributed_amd import ops


@pytest.mark.parametrize("E,H,I,rows,pays", [(64, 2048, 1024, 219, True), (64, 2048, 1024, 225, False), (64, 2048, 1024, 231, False),
                                             (64, 2048, 1024, 440, True), (16, 2048, 1408, 620, False), (32, 1024, 512, 470, False),
                                             (32, 1024, 512, 450, True), (8, 4096, 14336, 440, True), (8, 4096, 14336, 1025, True),
                                             (8, 4096, 14336, 200, False), (8, 1024, 512, 360, False)])
def test_rounds_opened_by_few_experts_count(E, H, I, rows, pays):
    assert ops._moe_wide_pays(E * rows, E, -(-I // 128), H, -(-H // 256), I) is pays
