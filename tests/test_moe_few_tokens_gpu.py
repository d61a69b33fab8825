"""Routed experts of few tokens: the K-split kernel's steps asked for ahead, from a column of each workgroup's own, and
the sizes at which 8-bit weights take it."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def experts(T, E, k, H, I, fp8, dt):
    torch.manual_seed(T + H + I)
    x = torch.randn(T, H, device=DEV).to(dt) * 0.5
    w13, w2 = torch.randn(E, 2 * I, H, device=DEV) * H ** -0.5, torch.randn(E, H, I, device=DEV) * I ** -0.5
    s13 = s2 = None
    if fp8:
        s13, s2 = w13.abs().amax(dim=(1, 2)) / 448, w2.abs().amax(dim=(1, 2)) / 448
        w13, w2 = (w13 / s13.view(E, 1, 1)).to(torch.float8_e4m3fn), (w2 / s2.view(E, 1, 1)).to(torch.float8_e4m3fn)
    else:
        w13, w2 = w13.to(dt), w2.to(dt)
    tw, ids = R.moe_topk_softmax(torch.randn(T, E, device=DEV), k, True)
    return x, w13, w2, tw, ids, s13, s2


def check(args, dt):
    out, ref = ops.fused_moe(*args), R.fused_moe(*args)
    # the activations between the products and the result are rounded to dt in both: a few units of the largest magnitude
    torch.testing.assert_close(out.float(), ref.float(), rtol=0, atol=6 * torch.finfo(dt).eps * float(ref.float().abs().max()))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T", [1, 5, 67])
@pytest.mark.parametrize("H,I", [(128, 128), (512, 640), (2176, 2688), (640, 2048)])
def test_steps_asked_for_ahead(monkeypatch, dt, fp8, T, H, I):
    """From no step for three of the four waves to several rounds of the ring, with and without a remainder; under a full
    tile of tokens, and several tiles."""
    monkeypatch.setenv("VDA_MOE_ROWS_FORM", "0")
    check(experts(T, 4, 2, H, I, fp8, dt), dt)


@pytest.mark.parametrize("T,E,k,H,I", [(1, 8, 2, 4096, 1024), (2, 8, 2, 4096, 6400), (4, 8, 2, 4096, 4096), (5, 8, 2, 4096, 4096)])
def test_either_side_of_the_rule(monkeypatch, T, E, k, H, I):
    """The form the sizes pick is, within rounding, what every other form gives."""
    args = experts(T, E, k, H, I, True, torch.bfloat16)
    for form in ("-1", "0", "1", "2"):
        monkeypatch.setenv("VDA_MOE_ROWS_FORM", form)
        check(args, torch.bfloat16)


def test_the_rule(monkeypatch):
    monkeypatch.delenv("VDA_MOE_ROWS_FORM", raising=False)
    form = ops.moe_rows_form
    assert form(2, 8, 4096, 1, 14336) == 0 and form(2, 8, 14336, 1, 4096) != 0 and form(4, 8, 14336, 1, 4096) == 0
    assert form(16, 64, 1024, 1, 2048) == 0 and form(32, 64, 1024, 1, 2048) != 0 and form(10, 8, 4096, 1, 14336) != 0
    assert form(2, 8, 4096, 2, 14336) == 0


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,k", [(95, 2), (96, 2), (64, 3), (1023, 1), (700, 3)])
def test_large_experts_from_tiles(monkeypatch, dt, T, k):
    """Experts of 264 MiB on both sides of 192 pairs, some of another rank, rows of a wider tensor: as the grouped kernel has it,
    within rounding; and replayed with other tokens."""
    x, w13, w2, tw, ids, _, _ = experts(T, 8, k, 4096, 1408, False, dt)
    assert ops.moe_grouped_limit(x, w13, w2) == 191
    x = torch.cat([x, x], 1)[:, :4096]
    ids[::5, 0] = -1

    def run():
        return ops.fused_moe(x, w13, w2, tw, ids)
    g = torch.cuda.CUDAGraph()
    run()
    with torch.cuda.graph(g):
        held = run()
    for _ in range(3):
        x.copy_(torch.randn_like(x) * 0.5)
        g.replay()
        out = run()
        monkeypatch.setenv("VDA_MOE_GROUPED_MAX_PAIRS_LARGE", "4096")
        monkeypatch.setenv("VDA_MOE_GROUPED_MAX_PAIRS", "4096")
        ref = run()
        monkeypatch.undo()
        atol = 6 * torch.finfo(dt).eps * float(ref.float().abs().max())      # (as above)
        torch.testing.assert_close(out.float(), ref.float(), rtol=0, atol=atol)
        torch.testing.assert_close(held.float(), ref.float(), rtol=0, atol=atol)
