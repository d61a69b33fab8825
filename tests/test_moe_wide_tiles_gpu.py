"""256 x 256 tiles of 16-bit experts (ops/csrc/gemm_tile.hip moe_wide_gemm_kernel) where they can go wrong: experts with no
row, one row, a row more or less than a fragment, half a tile and a whole tile, widths that end inside a tile, one unit of K,
pairs of another rank, and the block -> tile map at odd tile counts.

Tolerance: products are exact in the fp32 accumulator up to its own rounding; three results are rounded to 16 bits (the
activated middle, the weighted row of a pair, the sum over pairs), each by at most u = 2^-9 (bfloat16) or 2^-12 (float16) of
its size, so the result is within 3 u of the exact one in norm, plus u for the fast exp of the activation.  A single row has few
elements: 4 times that."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def at_any_cost(request, monkeypatch):
    """The kernel's tests take it wherever it can run, also where its tiles would leave the chip idle."""
    if "cost" not in request.node.name:
        monkeypatch.setattr(ops, "_moe_wide_pays", lambda *a: True)


def _routing(counts, k, g):
    """ids [T, k] in which expert e appears counts[e] times (in mixed order; -1 fills the last token)."""
    ids = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(ids.numel(), generator=g)]
    ids = torch.cat([ids, torch.full((-ids.numel() % k,), -1)])
    return ids.view(-1, k).to(torch.int32)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,k,H,I,gated", [
    ([1, 0, 15, 16, 17, 127, 128, 129, 255, 256, 257, 801], 1, 64, 64, True),
    ([129], 1, 128, 192, True),                       # the fewest rows, one tile cut in its second half
    ([1025, 383], 2, 320, 448, True),
    ([513, 0, 1, 272, 1400, 31], 2, 192, 320, False),
    ([200] * 9, 4, 576, 1088, True),                  # 9 x 9 and 9 x 3 tiles: eighths that do not come out even
    ([700, 705] * 20, 3, 128, 1152, True),            # whole rounds of 512 tiles and a rest
    ([287, 288, 289, 320, 321, 576, 577, 865, 33, 64, 65, 96, 1153], 1, 64, 192, True),      # either side of 288 rows, and of 32 of them
    ([224, 193, 160, 225, 97, 320], 1, 192, 320, False),      # each number of fragments
])
def test_wide_tiles(monkeypatch, dt, counts, k, H, I, gated):
    monkeypatch.setenv("VDA_MOE_GROUPED_MAX_PAIRS", "0")
    g = torch.Generator().manual_seed(len(counts) * H + I)
    ids = _routing(counts, k, g)
    T, E = ids.shape[0], len(counts)
    x = (torch.randn(T, H, generator=g) * 0.5).to(dt).to(DEV)
    w13 = (torch.randn(E, (2 if gated else 1) * I, H, generator=g) * 0.08).to(dt).to(DEV)
    w2 = (torch.randn(E, H, I, generator=g) * 0.08).to(dt).to(DEV)
    tw = torch.rand(T, k, generator=g).to(DEV) + 0.1
    ids = ids.to(DEV)
    assert ops._moe_wide_ok(x, w13, w2, T * k)
    out = ops.fused_moe(x, w13, w2, tw, ids, gated=gated).double()
    ref = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in range(E):
        tok, slot = torch.where(ids == e)
        h = x[tok].double() @ w13[e].double().t()
        h = torch.nn.functional.silu(h[:, :I]) * h[:, I:] if gated else torch.nn.functional.silu(h)
        ref.index_add_(0, tok, (h @ w2[e].double().t()) * tw[tok, slot].double().unsqueeze(1))
    u = 2.0 ** (-9 if dt == torch.bfloat16 else -12)
    assert float((out - ref).norm() / ref.norm()) < 4 * u
    live = ref.norm(dim=1) > 0
    rows = (out - ref).norm(dim=1)[live] / ref.norm(dim=1)[live]
    assert float(rows.max()) < 16 * u
    assert float(out[~live].abs().sum()) == 0


def test_rule_and_the_other_tiles_agree(monkeypatch):
    """Where the rule does not take them the 128-row tiles run; both give the same rows up to the last bit of a rounding."""
    monkeypatch.setenv("VDA_MOE_GROUPED_MAX_PAIRS", "0")
    g = torch.Generator().manual_seed(3)
    E, H, I = 4, 256, 320
    w13 = (torch.randn(E, 2 * I, H, generator=g) * 0.08).to(torch.bfloat16).to(DEV)
    w2 = (torch.randn(E, H, I, generator=g) * 0.08).to(torch.bfloat16).to(DEV)
    took = {}
    for rows in (128, 129, 232, 233, 351, 352, 600):
        T = rows * E
        x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(DEV)
        ids = torch.randint(0, E, (T, 1), generator=g).to(torch.int32).to(DEV)
        tw = torch.ones(T, 1, device=DEV)
        took[rows] = ops._moe_wide_ok(x, w13, w2, T)
        out = ops.fused_moe(x, w13, w2, tw, ids)
        with monkeypatch.context() as m:
            m.setattr(ops, "_moe_wide_ok", lambda *a: False)
            other = ops.fused_moe(x, w13, w2, tw, ids)
        # the middle may round differently in a few places: 2 u of a row's norm in any element
        lim = 2 * 2.0 ** -9 * other.float().norm(dim=1, keepdim=True)
        assert bool(((out.float() - other.float()).abs() <= lim).all())
    assert took == {128: False, 129: True, 232: True, 233: False, 351: False, 352: True, 600: True}


@pytest.mark.parametrize("E,k,H,I,rows,wide", [(8, 2, 1024, 512, 360, False),        # fewer tiles than CUs
                                               (32, 4, 1024, 512, 160, False),       # one round of either
                                               (64, 8, 1024, 512, 160, True), (64, 8, 1024, 512, 440, True)])
def test_the_cost_of_rounds_decides(monkeypatch, E, k, H, I, rows, wide):
    """By the launch that is made; and the result is that of the other tiles (see above)."""
    monkeypatch.setenv("VDA_MOE_GROUPED_MAX_PAIRS", "0")
    g = torch.Generator().manual_seed(rows)
    T = rows * E // k
    gd = torch.Generator(device=DEV).manual_seed(rows)
    w13 = (torch.randn(E, 2 * I, H, generator=gd, device=DEV) * 0.08).to(torch.bfloat16)
    w2 = (torch.randn(E, H, I, generator=gd, device=DEV) * 0.08).to(torch.bfloat16)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(DEV)
    tw, ids = ops.moe_topk_softmax(torch.randn(T, E, generator=g).to(DEV), k)
    out, took, call = [], [], ops.N.call
    for force in (None, True, False):
        with monkeypatch.context() as m:
            if force is not None:
                m.setattr(ops, "_moe_wide_pays", lambda *a: force)
            m.setattr(ops.N, "call", lambda name, *a: (took.append(a[-6]) if name == "vda_tile_gemm" else None, call(name, *a))[1])
            out.append(ops.fused_moe(x, w13, w2, tw, ids).float())
    assert took == [256 if wide else 128] * 2 + [256] * 2 + [128] * 2
    # pairs' rows round to bfloat16 in both, k of them are summed: 2 u of a pair's row each, of k rows of random sign
    lim = 2 * 2.0 ** -9 * k * out[2].norm(dim=1, keepdim=True)
    assert bool(((out[1] - out[2]).abs() <= lim).all())
    assert torch.equal(out[0], out[1 if wide else 2])
