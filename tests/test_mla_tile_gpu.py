"""Latent attention over LDS-staged tiles (ops/csrc/mla_tile.hip: caches of 576-value rows) against the 32-bit form
in PyTorch: edges of the 32-key tiles and of the 32- and 128-column blocks, pages of every size it takes, keys cut
into pieces, windows and sinks, rows of a page that hold no key."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV, DK, DV = "cuda", 576, 512


def _batch(new, total, page, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    pages = [-(-t // page) for t in total]
    perm = torch.randperm(sum(pages) + 3, generator=g).int()
    table = torch.zeros((len(new), max(pages) + 1), dtype=torch.int32)
    kc = torch.full((sum(pages) + 3, page, DK), 448. if dtype == torch.float8_e4m3fn else 1e4)              # what no key of a sequence may bring in
    at = 0
    for s, (n, t) in enumerate(zip(new, total)):
        table[s, :pages[s]] = perm[at:at + pages[s]]
        at += pages[s]
        pos = torch.arange(t)
        kc[table[s, pos // page].long(), pos % page] = torch.randn(t, DK, generator=g)
    kc = kc.to(dtype)
    vt = kc[..., :DV].transpose(1, 2).contiguous()
    starts = torch.tensor([0] + new).cumsum(0).int()
    return [t.to(DEV) for t in (kc, vt, table, torch.tensor(total, dtype=torch.int32), starts)]


CASES = [  # new tokens, keys in all, heads
    ([1, 1, 1, 1], [1, 31, 32, 33], 16),                # one wave's columns, tile edges
    ([1], [1500], 16),                                   # pieces of one long sequence
    ([1, 1, 1], [40, 700, 2100], 32),                    # ragged pieces
    ([1, 2, 1], [64, 97, 300], 20),                      # columns that fill no block; two tokens in a step
    ([1, 1], [129, 4000], 128),                          # decoding with a column block per token
    ([5, 130, 33], [5, 130, 400], 16),                   # prompts, one continued: causal edges inside a tile
    ([9], [9], 128),
    ([7, 1], [260, 33], 40),
]


@pytest.mark.parametrize("new,total,H", CASES)
@pytest.mark.parametrize("page,dtype,fp8", [(16, torch.bfloat16, False), (64, torch.float16, False),
                                            (16, torch.float16, True), (32, torch.bfloat16, True)])
def test_tiles_match_fp32(new, total, H, page, dtype, fp8):
    kc, vt, table, lens, starts = _batch(new, total, page, torch.float8_e4m3fn if fp8 else dtype, H + len(new))
    kv_scale = 0.75 if fp8 else 1.0
    for window, with_sink in ((0, False), (100, True)):
        q = torch.randn(sum(new), H, DK, device=DEV).to(dtype)
        sink = torch.randn(H, device=DEV) if with_sink else None
        out = torch.empty(sum(new), H, DV, device=DEV, dtype=dtype)
        ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, max(new), 1, kv_scale=kv_scale, window=window, sink=sink)
        want = R.mla_attention(q, kc, vt, table, lens, starts, 192 ** -0.5, kv_scale, window, sink)
        # weights and result are rounded to 16 bits: 2^-9 (bf16) / 2^-12 (fp16) of values up to ~4, three times over
        eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
        torch.testing.assert_close(out.float(), want.float(), atol=12 * eps, rtol=2 * eps)


def test_growing_scores_rescale_the_sums():
    """Scores that grow along the keys by far more than the lag allowed to the running maximum."""
    kc, vt, table, lens, starts = _batch([3], [500], 16, torch.bfloat16, 5)
    q = torch.ones(3, 16, DK, device=DEV, dtype=torch.bfloat16)
    for pos in range(500):
        kc[table[0, pos // 16].long(), pos % 16, 0] = pos * 0.5
    vt = kc[..., :DV].transpose(1, 2).contiguous()
    out = torch.empty(3, 16, DV, device=DEV, dtype=torch.bfloat16)
    ops.mla_attention(out, q, kc, vt, table, lens, starts, 0.5, 3, 1)
    want = R.mla_attention(q, kc, vt, table, lens, starts, 0.5)
    torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("H", [16, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn])
def test_rows_without_keys(H, dtype):
    """Padded sequences (no keys) among others, with pieces: their rows are merged from what was written for them alone.  Tokens
    before their sequence's first key (fewer keys than new tokens), in one piece and in several: zero."""
    kc, vt, table, lens, starts = _batch([1, 1, 1], [40, 700, 2100], 16, dtype, 8)
    lens[1] = 0
    q = torch.randn(3, H, DK, device=DEV).to(torch.bfloat16)
    out = torch.full((3, H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
    for fill in (float("inf"), 0.0, -1.0):               # whatever the pieces' workspace held before
        torch.full((3 * H * 16 * (DV + 1) * 2,), fill, device=DEV)
        ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, 1, 8)
        assert bool((out[1] == 0).all())
    live = torch.tensor([0, 2], device=DEV)
    want = R.mla_attention(q[live], kc, vt, table[live], lens[live], torch.tensor([0, 1, 2], dtype=torch.int32, device=DEV), 192 ** -0.5)
    torch.testing.assert_close(out[live].float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)
    for total, width in (([9, 40], 4), ([9, 900], 90)):  # a table of one piece, and of several
        kc, vt, table, lens, starts = _batch([20, 3], [20, total[1]], 16, dtype, 9)
        lens[0] = total[0]
        wide = torch.zeros((2, width), dtype=torch.int32, device=DEV)
        wide[:, :min(width, table.shape[1])] = table[:, :width]
        q = torch.randn(23, H, DK, device=DEV).to(torch.bfloat16)
        out = torch.full((23, H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.mla_attention(out, q, kc, vt, wide, lens, starts, 192 ** -0.5, 20, 1)
        assert bool((out[:11] == 0).all()) and bool(out.isfinite().all())
        want = R.mla_attention(q[11:], kc, vt, wide, lens, torch.tensor([0, 9, 12], dtype=torch.int32, device=DEV), 192 ** -0.5)
        torch.testing.assert_close(out[11:].float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("H,new,dtype", [(16, 1, torch.bfloat16), (128, 1, torch.float16), (40, 3, torch.bfloat16),
                                         (16, 1, torch.float8_e4m3fn)])
def test_a_sequence_does_not_see_its_neighbours_lengths(H, new, dtype):
    """Where its keys are cut depends on the batch's size and the table's width, not on how long the others are: the same bits."""
    S, width = 5, 300
    qd = torch.bfloat16 if dtype == torch.float8_e4m3fn else dtype
    first = None
    for others in ([40, 50, 60, 70], [4000, 3500, 4100, 2900], [1, 0, 2000, 3]):
        total = [new + 1700] + [new + t if t else 0 for t in others]
        kc, vt, table, lens, starts = _batch([new] * S, total, 16, dtype, 3)
        g = torch.Generator().manual_seed(4)
        rows = torch.randn(total[0], DK, generator=g).to(DEV).to(kc.dtype)
        pos = torch.arange(total[0], device=DEV)
        kc[table[0, pos // 16].long(), pos % 16] = rows
        wide = torch.zeros((S, width), dtype=torch.int32, device=DEV)
        wide[:, :table.shape[1]] = table
        q = torch.randn(new, H, DK, generator=g).to(qd).to(DEV).repeat(S, 1, 1)
        out = torch.empty(S * new, H, DV, device=DEV, dtype=qd)
        ops.mla_attention(out, q, kc, kc[..., :DV].transpose(1, 2).contiguous(), wide, lens, starts, 192 ** -0.5, new, 8)
        first = out[:new].clone() if first is None else first
        assert torch.equal(out[:new], first)


@pytest.mark.parametrize("new,total,H", [([1] * 6, [9, 64, 300, 700, 1500, 2900], 128), ([1] * 3, [40, 900, 3000], 16),
                                         ([260, 90], [260, 700], 16)])
@pytest.mark.parametrize("dtype,fp8", [(torch.bfloat16, False), (torch.float16, False), (torch.bfloat16, True)])
def test_error_is_that_of_rounding_the_result(new, total, H, dtype, fp8):
    """Weights keep more than 16 bits (also where the maximum that they are relative to lags): against 64 bits the result is off by its own
    rounding and little else.  With weights of 16 bits it is 1.07 (the largest exact) to 1.25 times that."""
    kc, vt, table, lens, starts = _batch(new, total, 16, torch.float8_e4m3fn if fp8 else dtype, 11)
    q = torch.randn(sum(new), H, DK, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    out = torch.empty(sum(new), H, DV, device=DEV, dtype=dtype)
    ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, max(new), 1)
    want, at = torch.empty(sum(new), H, DV, dtype=torch.float64, device=DEV), 0
    for s, (n, t) in enumerate(zip(new, total)):
        pos = torch.arange(t, device=DEV)
        k = kc[table[s, pos // 16].long(), pos % 16].double()
        sc = q[at:at + n].double().reshape(-1, DK) @ k.t() * 192 ** -0.5
        sc = sc.view(n, H, t).masked_fill(pos > (t - n + pos[:n])[:, None, None], float("-inf"))
        want[at:at + n] = torch.softmax(sc, -1) @ k[:, :DV]
        at += n
    off, rounding = (out.double() - want).norm(), (want.to(dtype).double() - want).norm()
    assert float(off / rounding) < 1.02


@pytest.mark.parametrize("new,keys,H", [(1, 9000, 16), (1, 2049, 128), (3, 4100, 16)])
def test_one_long_sequence_in_many_pieces(new, keys, H):
    """Alone in its batch a sequence is cut into up to 64 pieces; behind a table that could hold far more, too."""
    kc, vt, table, lens, starts = _batch([new], [keys], 16, torch.bfloat16, 12)
    wide = torch.zeros((1, 2048), dtype=torch.int32, device=DEV)
    wide[:, :table.shape[1]] = table
    blocks = -(-new * H // (128 if new * H > 32 else 32))
    assert ops.N.lib().vda_mla_splits(1, new, H, DK, 16, 2048, new, 192 ** -0.5, 1) == 64 and blocks <= 2
    q = torch.randn(new, H, DK, device=DEV).to(torch.bfloat16)
    out = torch.empty(new, H, DV, device=DEV, dtype=torch.bfloat16)
    ops.mla_attention(out, q, kc, vt, wide, lens, starts, 192 ** -0.5, new, 1)
    want = R.mla_attention(q, kc, vt, wide, lens, starts, 192 ** -0.5)
    torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("page,scale", [(8, 192 ** -0.5), (24, 192 ** -0.5), (16, -(192 ** -0.5))])
@pytest.mark.parametrize("new,total,H", [([1, 1], [40, 700], 16), ([5, 70], [5, 130], 16)])
@pytest.mark.parametrize("fp8", [False, True])
def test_what_the_tiles_do_not_take(page, scale, new, total, H, fp8):
    """Pages off a power of two or below 16 tokens, and scales below zero, stay with the kernels of mla.hip."""
    kc, vt, table, lens, starts = _batch(new, total, page, torch.float8_e4m3fn if fp8 else torch.bfloat16, 13)
    q = torch.randn(sum(new), H, DK, device=DEV).to(torch.bfloat16)
    out = torch.empty(sum(new), H, DV, device=DEV, dtype=torch.bfloat16)
    for splits in (1, 3):
        ops.mla_attention(out, q, kc, vt, table, lens, starts, scale, max(new), splits)
        want = R.mla_attention(q, kc, vt, table, lens, starts, scale)
        torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


def _ragged(n, mean):
    return [max(1, int(mean * (0.25 + 1.5 * ((0.618 * i + 0.37) % 1)))) for i in range(n)]


@pytest.mark.parametrize("S,new,prefix,H,window", [
    (16, 1, 900, 16, 0), (17, 1, 300, 16, 0), (64, 1, 200, 128, 0), (65, 1, 200, 40, 90), (190, 1, 120, 32, 0), (260, 1, 60, 128, 0),       # decoding
    (2, 150, 0, 128, 0), (8, 90, 200, 32, 0), (16, 30, 100, 16, 50), (17, 40, 60, 128, 0), (70, 9, 30, 128, 0), (260, 3, 20, 64, 0),      # prompts
    (3, 5, 1500, 16, 700), (5, 12, 2000, 16, 0), (6, 3, 700, 128, 100)])                                            # blocks and pieces
def test_every_column_block_and_piece_has_its_workgroup(S, new, prefix, H, window):
    """Workgroups are numbered over the work that the lengths give: sorted (up to 16 sequences), two halves (up to 256), by column
    block (sequences alike, or more); among them sequences without a new token."""
    news = [1] * S if new == 1 else _ragged(S, new)
    if S > 4:
        news[1] = news[S - 2] = 0
    total = [n + p for n, p in zip(news, _ragged(S, prefix)[::-1])] if prefix else list(news)
    kc, vt, table, lens, starts = _batch(news, total, 16, torch.bfloat16, S)
    q = torch.randn(sum(news), H, DK, device=DEV).to(torch.bfloat16)
    out = torch.full((sum(news), H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, max(news), 8, window=window)
    want = R.mla_attention(q, kc, vt, table, lens, starts, 192 ** -0.5, 1.0, window)
    torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("new,total,H,window", [([264], [534], 1, 2), ([264, 1, 0, 40], [534, 90, 7, 41], 1, 2), ([659] + [3] * 23, [3583] + [3] * 23, 1, 1),
                                                ([300], [900], 2, 33), ([200], [700], 3, 1)])
def test_windows_of_blocks_of_many_tokens(new, total, H, window):
    """With one head a column block is 128 tokens: under a window it has up to five key steps more than a last block of one token, and
    as many more pieces."""
    kc, vt, table, lens, starts = _batch(new, total, 16, torch.bfloat16, H)
    q = torch.randn(sum(new), H, DK, device=DEV).to(torch.bfloat16)
    out = torch.full((sum(new), H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, max(new), 8, window=window)
    want = R.mla_attention(q, kc, vt, table, lens, starts, 192 ** -0.5, 1.0, window)
    torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("S,H,new", [(1, 16, 1), (7, 16, 1), (12, 16, 1), (13, 16, 1), (6, 16, 2), (3, 5, 6), (1, 128, 1), (6, 128, 1), (7, 128, 1), (6, 40, 3)])
@pytest.mark.parametrize("fp8", [False, True])
def test_few_sequences_piece_by_piece(S, H, new, fp8):
    """Sequences of one column block, either side of where workgroups look through the lengths: pieces of unlike numbers, one sequence without
    a new token, and rows that an unused piece must leave to the others."""
    news = [new] * S
    if S > 3:
        news[2] = 0
    total = [n + p for n, p in zip(news, _ragged(S, 1300))]
    kc, vt, table, lens, starts = _batch(news, total, 16, torch.float8_e4m3fn if fp8 else torch.bfloat16, S + H)
    q = torch.randn(sum(news), H, DK, device=DEV).to(torch.bfloat16)
    for window in (0, 70):
        out = torch.full((sum(news), H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, new, 8, window=window)
        want = R.mla_attention(q, kc, vt, table, lens, starts, 192 ** -0.5, 1.0, window)
        torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("S,H,new", [(3, 16, 51), (7, 16, 60), (2, 128, 45), (5, 1, 800)])
def test_ragged_prompts_that_run_at_once(S, H, new):
    """As many column blocks as CUs at most: by block, then sequence, whatever the lengths; a sequence without a new token among them."""
    news = _ragged(S, new)
    if S > 3:
        news[1] = 0
    kc, vt, table, lens, starts = _batch(news, news, 16, torch.bfloat16, S + H)
    q = torch.randn(sum(news), H, DK, device=DEV).to(torch.bfloat16)
    out = torch.full((sum(news), H, DV), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.mla_attention(out, q, kc, vt, table, lens, starts, 192 ** -0.5, max(news), 1)
    want = R.mla_attention(q, kc, vt, table, lens, starts, 192 ** -0.5)
    torch.testing.assert_close(out.float(), want.float(), atol=12 * 2.0 ** -9, rtol=2.0 ** -8)
