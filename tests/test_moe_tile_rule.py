"""Which 16-bit expert layers take 256-row tiles (ops._moe_wide_pays): where single experts past a tile's rows open another round over
the CUs, they do not.  Layers by experts, hidden and intermediate width, and rows an expert; times in the rule's comment."""
import pytest
import torch

from vllm_distributed_amd import envs, ops


@pytest.mark.parametrize("E,H,I,rows,pays", [(64, 2048, 1024, 219, True), (64, 2048, 1024, 225, False), (64, 2048, 1024, 231, False),
                                             (64, 2048, 1024, 440, True), (16, 2048, 1408, 620, False), (32, 1024, 512, 470, False),
                                             (32, 1024, 512, 450, True), (8, 4096, 14336, 440, True), (8, 4096, 14336, 1025, True),
                                             (8, 4096, 14336, 200, False), (8, 1024, 512, 360, False)])
def test_rounds_opened_by_few_experts_count(E, H, I, rows, pays):
    assert ops._moe_wide_pays(E * rows, E, -(-I // 128), H, -(-H // 256), I) is pays


@pytest.mark.parametrize("pairs,large,limit", [(None, None, 191), ("4096", None, 4096), ("64", None, 64), (None, "500", 500),
                                               ("4096", "500", 500), ("300", "500", 300)])
def test_a_limit_that_is_set_holds_for_large_experts(monkeypatch, pairs, large, limit):
    for name, value in (("VDA_MOE_GROUPED_MAX_PAIRS", pairs), ("VDA_MOE_GROUPED_MAX_PAIRS_LARGE", large)):
        monkeypatch.delenv(name, raising=False)
        if value is not None:
            monkeypatch.setenv(name, value)
        assert envs.is_set(name) == (value is not None)
    x, w13, w2 = (torch.empty(s, dtype=torch.bfloat16, device="meta") for s in ((1, 4096), (8, 28672, 4096), (8, 4096, 14336)))
    assert ops.moe_grouped_limit(x, w13, w2) == limit
    small = [torch.empty(s, dtype=torch.bfloat16, device="meta") for s in ((8, 1024, 1024), (8, 1024, 512))]
    assert ops.moe_grouped_limit(x, *small) == int(pairs or 2048)


@pytest.mark.parametrize("E,H,I,limit", [(8, 4096, 1408, 191), (8, 4096, 1280, 383), (8, 4096, 1024, 383), (7, 4096, 1024, 2048), (16, 2048, 1024, 383),
                                         (64, 1536, 512, 191), (32, 1024, 1408, 2048), (8, 1024, 5632, 2048), (64, 1024, 1024, 191)])
def test_which_experts_are_large(monkeypatch, E, H, I, limit):
    """Where tiles lead, by the measurements beside the rule: at either side of its lines in bytes and in width."""
    for name in ("VDA_MOE_GROUPED_MAX_PAIRS", "VDA_MOE_GROUPED_MAX_PAIRS_LARGE"):
        monkeypatch.delenv(name, raising=False)
    x, w13, w2 = (torch.empty(s, dtype=torch.bfloat16, device="meta") for s in ((1, H), (E, 2 * I, H), (E, H, I)))
    assert ops.moe_grouped_limit(x, w13, w2) == limit


@pytest.mark.parametrize("pairs,E,rows,depth,split", [(6, 8, 4096, 14336, True), (4, 8, 7168, 4096, True), (8, 32, 4096, 4096, False), (9, 32, 4096, 4096, True),
                                                      (8, 16, 4096, 6400, True), (32, 128, 768, 2048, True), (12, 60, 2048, 1408, False),
                                                      (8, 60, 2048, 1408, True), (2, 8, 14336, 4096, False), (8, 256, 2048, 7168, True)])
def test_few_pairs_of_8_bit_experts(monkeypatch, pairs, E, rows, depth, split):
    """The K-split form where the workgroups of the experts that are chosen are too few for the other, or more than its first wave."""
    monkeypatch.delenv("VDA_MOE_ROWS_FORM", raising=False)
    assert (ops.moe_rows_form(pairs, E, rows, 1, depth) == 0) is split


@pytest.mark.parametrize("E,H,I,rows,wide", [(64, 2048, 1024, 128, False), (64, 2048, 1024, 129, True), (64, 2048, 1024, 300, True),     # 512 and 512 tiles
                                             (8, 4096, 14336, 256, True), (8, 3840, 14336, 256, False),       # 128 and 120 in the second product
                                             (8, 4096, 8192, 256, True), (8, 4096, 8064, 256, False),         # 512 and 504 in the first
                                             (16, 1024, 4096, 300, False), (32, 1024, 512, 450, True)])
def test_layers_of_many_tiles_take_the_wide_ones_at_any_rows(E, H, I, rows, wide):
    x, w13, w2 = (torch.empty(s, dtype=torch.bfloat16, device="meta") for s in ((E * rows, H), (E, 2 * I, H), (E, H, I)))
    assert ops._moe_wide(x, w13, w2, E * rows, -(-I // 128), H, -(-H // 256), I) is wide
    assert not ops._moe_wide(x, w13.to(torch.float8_e4m3fn), w2, E * rows, -(-I // 128), H, -(-H // 256), I)
