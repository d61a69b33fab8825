"""Whether a batch of prompts takes the wide form (vda_prefill_form answers 0): batches on either side of the lines, by the measurements beside them."""
import pytest

from vllm_distributed_amd.ops import native as N

pytestmark = pytest.mark.skipif(not N.is_available(), reason="libvda_ops.so is not built")


def _wide(heads, new, known=True):
    Hq, Hkv, D = heads
    return N.value("vda_prefill_form", len(new), sum(new), Hq, Hkv, D, max(new) + 300, max(new) if known else 0) == 0


@pytest.mark.parametrize("heads,new,wide", [
    # heads of 128, a long prompt among short ones: as many of them as it saves for
    ((32, 8, 128), [2000] + [10] * 100, True), ((32, 8, 128), [2000] + [15] * 250, True), ((32, 8, 128), [4000] + [10] * 400, True),
    ((32, 8, 128), [2000] + [10] * 443, True), ((32, 8, 128), [2000] + [10] * 444, False), ((32, 8, 128), [2000] + [10] * 1000, False),
    ((32, 8, 128), [1000] + [8] * 100, True), ((32, 8, 128), [1000] + [8] * 200, False), ((32, 8, 128), [500] + [8] * 100, False),
    ((64, 8, 128), [3000] + [2] * 400, True), ((64, 8, 128), [2000] + [10] * 500, False),
    ((32, 32, 128), [1500] + [10] * 130, True), ((32, 32, 128), [1000] + [8] * 200, False),
    # prompts of one length
    ((32, 8, 128), [20] * 160, False), ((32, 8, 128), [31] * 80, False), ((32, 8, 128), [32] * 80, True), ((64, 8, 128), [15] * 200, False),
    ((64, 8, 128), [16] * 200, True), ((32, 32, 128), [39] * 60, False), ((32, 32, 128), [40] * 60, True),
    # too few tiles for half of the CUs
    ((32, 8, 128), [1000], False), ((32, 8, 128), [1024], True), ((8, 1, 128), [2000] + [10] * 100, False),
    # heads of 96 and 64: what they took before they had the form, where prompts do not fill its tiles
    ((24, 8, 96), [2000] + [10] * 100, False), ((24, 8, 96), [43] * 60, True), ((24, 8, 96), [41] * 60, False), ((32, 8, 64), [2000] + [10] * 100, False),
    ((32, 8, 64), [63] * 20, False), ((32, 8, 64), [64] * 32, True), ((32, 8, 64), [100] * 40, False), ((32, 8, 64), [192] * 40, True)])
def test_wide_form(heads, new, wide):
    assert _wide(heads, new) is wide


def test_a_longest_run_that_is_not_known():
    """The mean decides then; and a bound above the batch's tokens is one of all of them."""
    assert not _wide((32, 8, 128), [2000] + [10] * 100, known=False) and _wide((32, 8, 128), [32] * 80, known=False)
    ask = lambda longest: N.value("vda_prefill_form", 200, 3000, 32, 8, 128, 3000, longest) == 0
    assert ask(3000) and ask(1 << 40) and not ask(0)
    ask = lambda longest: N.value("vda_prefill_form", 1200, 3000, 32, 8, 128, 3000, longest) == 0
    assert not ask(3000) and not ask(1 << 40)
