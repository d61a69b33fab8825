"""Which decode calls of two parts are eight waves of one workgroup (ops.decode_parts_as_waves): short sequences alone."""
import pytest

from vllm_distributed_amd import ops


@pytest.mark.parametrize("splits,S,Hq,Hkv,D,q_len,keys,waves", [(2, 5, 32, 8, 128, 1, 640, True), (2, 32, 32, 8, 128, 1, 768, True),
                                                                (2, 5, 32, 8, 128, 1, 769, False), (2, 1, 32, 8, 128, 1, 32000, False),
                                                                (2, 33, 32, 8, 128, 1, 640, False), (3, 5, 32, 8, 128, 1, 640, False),
                                                                (2, 5, 16, 8, 256, 1, 640, False), (2, 5, 32, 8, 128, 5, 640, False)])
def test_rule(splits, S, Hq, Hkv, D, q_len, keys, waves):
    assert ops.decode_parts_as_waves(splits, S, Hq, Hkv, D, q_len, keys) is waves


def test_every_call_for_which_two_parts_are_asked_for_is_short():
    for S in range(1, 40):
        for keys in range(1, 3000, 7):
            if ops.decode_num_splits(S, 8, keys) == 2 and S * 8 <= 256:
                assert keys < 768
