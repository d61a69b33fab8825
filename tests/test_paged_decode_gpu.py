"""Decode attention (ops/csrc/attention.hip paged_decode_kernel) where it can go wrong: key counts around a step (32 keys of a
16-bit cache, 64 of an e4m3 one), around a step of each wave and of each part, empty sequences, windows and chunks that start
inside a page, 16 and 32 query columns, every head size and page size, and the longest-first order of large grids (equal
lengths, the most sequences that it ranks, one more).

Tolerance: a weight is rounded to 16 bits (unit u) under a sum that is not, the output once more: with weights that add up to
one an element moves by at most 2 u max|v|; fp32 sums and the bare exponential add a few 1e-6 of it (1e-5 here)."""
import zlib

import numpy as np
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
FP8 = torch.float8_e4m3fn
EDGES = [1, 31, 32, 33, 63, 64, 65, 128, 129, 255, 256, 257, 511, 513, 777]


def _check(lens, new, Hq, Hkv, D, BS, dt, fp8, nsplit, **kw):
    g = torch.Generator().manual_seed(len(lens) * D + BS + nsplit)
    S, T = len(lens), sum(new)
    need = [max(1, -(-n // BS)) for n in lens]
    order = torch.randperm(sum(need) + 3, generator=g)
    table = torch.zeros(S, max(need), dtype=torch.int32)
    at = 0
    for s, n in enumerate(need):
        table[s, :n] = order[at:at + n].to(torch.int32)
        at += n
    pages = order.numel()
    k = torch.randn(pages, Hkv, BS, D, generator=g).to(DEV)
    v = torch.randn(pages, Hkv, D, BS, generator=g).to(DEV)
    q = torch.randn(T, Hq, D, generator=g).to(dt).to(DEV)
    ks, vs = (0.5, 0.25) if fp8 else (1.0, 1.0)
    kc, vc = (k.to(FP8), v.to(FP8)) if fp8 else (k.to(dt), v.to(dt))
    starts = torch.tensor([0] + new).cumsum(0).to(torch.int32).to(DEV)
    sl, table = torch.tensor(lens, dtype=torch.int32, device=DEV), table.to(DEV)
    out = torch.empty(T, Hq, D, dtype=dt, device=DEV)
    ops.paged_attention_decode(out, q, kc, vc, table, sl, starts, D ** -0.5, num_splits=nsplit, max_q_len=max(new),
                               k_scale=ks, v_scale=vs, **kw)
    chunk = kw.pop("chunk", 0)
    vis = (lambda pos, key: ((pos // chunk) == (key // chunk)).expand(Hq, -1, -1)) if chunk else None
    kf, vf = kc.float() * ks, vc.float() * vs
    live = [s for s in range(S) if lens[s] > 0]
    ref = torch.zeros(T, Hq, D, device=DEV)
    rows = torch.cat([torch.arange(int(starts[s]), int(starts[s + 1])) for s in live]).to(DEV)
    n_live = torch.tensor([0] + [new[s] for s in live]).cumsum(0).to(torch.int32).to(DEV)
    ref[rows] = R.paged_attention(q.float()[rows], kf, vf, table[live], sl[live], n_live, D ** -0.5, visible=vis, **kw)
    u = 2.0 ** (-9 if dt == torch.bfloat16 else -12)
    assert float((out.float() - ref).abs().max()) <= (2 * u + 1e-5) * float(vf.abs().max())


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,BS,Hq,Hkv", [(64, 16, 8, 2), (64, 64, 4, 4), (128, 16, 16, 1), (128, 32, 14, 2), (128, 64, 8, 8),
                                          (96, 16, 6, 2), (192, 32, 4, 1), (256, 16, 4, 2)])
@pytest.mark.parametrize("nsplit", [1, 3, 16])
def test_key_counts(D, BS, Hq, Hkv, fp8, nsplit):
    if fp8 and D not in (64, 128):
        pytest.skip("e4m3 caches: head sizes 64 and 128")
    _check(EDGES + [0], [1] * (len(EDGES) + 1), Hq, Hkv, D, BS, torch.bfloat16, fp8, nsplit)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("kw", [dict(window=1), dict(window=100), dict(chunk=96), dict(softcap=5.0)])
@pytest.mark.parametrize("D,Hq,Hkv", [(64, 8, 2), (128, 32, 4)])
def test_masks_and_several_tokens(D, Hq, Hkv, kw, fp8):
    lens = [max(n, 4) for n in EDGES] + [1500]
    _check(lens, [1 + i % 4 for i in range(len(lens))], Hq, Hkv, D, 16, torch.float16, fp8, 2, **kw)


@pytest.mark.parametrize("S,Hkv,nsplit", [(65, 8, 1), (256, 3, 1), (257, 2, 1), (100, 2, 3)])
def test_longest_first(S, Hkv, nsplit):
    lens = [(EDGES * 20)[i] if i % 3 else 200 for i in range(S)]
    _check(lens, [1] * S, 2 * Hkv, Hkv, 128, 16, torch.bfloat16, True, nsplit)


# grids above 512 workgroups: lengths alike (their own order), all within an eighth but one, and rows without keys
@pytest.mark.parametrize("S", [65, 129, 256])
@pytest.mark.parametrize("lens", [lambda i, S: 130, lambda i, S: 128 + i % 9, lambda i, S: 600 if i == S - 1 else 130,
                                  lambda i, S: 0 if i % 5 == 1 else 77])
def test_order_of_large_batches(S, lens):
    lens = [lens(i, S) for i in range(S)]
    _check(lens, [1] * S, 16, 8, 128, 16, torch.bfloat16, S == 129, 1)


# the merge of the parts: one wave's last count, four waves' first, the most; parts with and without keys
@pytest.mark.parametrize("nsplit", [2, 8, 9, 64])
@pytest.mark.parametrize("D", [64, 96, 128, 192, 256])
def test_merge_of_parts(D, nsplit):
    _check([1, 40, 300, 2100, 0], [1] * 5, 6, 2, D, 16, torch.bfloat16, False, nsplit)


# two parts of few sequences: eight waves of one workgroup (up to 256 of them), parts and a merge beyond and above 16 columns
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,Hq,Hkv,S", [(64, 4, 4, 17), (128, 16, 1, 17), (96, 6, 2, 17), (192, 4, 1, 17), (256, 4, 2, 17), (128, 8, 8, 32),
                                        (128, 8, 8, 33), (128, 32, 1, 17)])
def test_two_parts(D, Hq, Hkv, S, fp8):
    if fp8 and D not in (64, 128):
        pytest.skip("e4m3 caches: head sizes 64 and 128")
    for longest in (768, 1025):                                     # (eight waves up to 768 keys; parts and a merge beyond them too)
        lens = [min(n, longest) for n in ((EDGES + [0, 1025]) * 2)[:S]]
        _check(lens, [1] * S, Hq, Hkv, D, 16, torch.bfloat16, fp8, 2)
        if Hq // Hkv <= 4:
            _check([max(n, 4) for n in lens], [1 + i % 4 for i in range(S)], Hq, Hkv, D, 16, torch.float16, fp8, 2, window=300)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("D,BS,Hq,Hkv,nsplit", [(128, 16, 32, 8, 2), (128, 64, 8, 8, 1), (64, 32, 8, 2, 2), (256, 16, 4, 2, 1), (128, 16, 32, 8, 3)])
def test_tables_hold_anything_past_a_sequence(D, BS, Hq, Hkv, nsplit, fp8):
    """The first pages are asked for ahead of a sequence's length: what lies behind its last page (here the number of a page of NaN, in a
    row that is longer than the table) is read and not used."""
    if fp8 and D not in (64, 128):
        pytest.skip("e4m3 caches: head sizes 64 and 128")
    g = torch.Generator().manual_seed(D + BS)
    lens = [1, 15, 16, 17, 33, 64, 65, 250, 300, 513, 700]
    S, width = len(lens), 704 // BS
    need = [-(-n // BS) for n in lens]
    pages = torch.randperm(sum(need), generator=g).to(torch.int32)
    nan = sum(need)
    wide = torch.full((S, width + 9), nan, dtype=torch.int32)
    at = 0
    for s, n in enumerate(need):
        wide[s, :n] = pages[at:at + n]
        at += n
    dt = FP8 if fp8 else torch.bfloat16
    k, v = torch.randn(nan + 1, Hkv, BS, D, generator=g), torch.randn(nan + 1, Hkv, D, BS, generator=g)
    k[nan], v[nan] = float("nan"), float("nan")
    q = torch.randn(S, Hq, D, generator=g).to(torch.bfloat16).to(DEV)
    starts = torch.arange(S + 1, dtype=torch.int32, device=DEV)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    kc, vc = k.to(dt).to(DEV), v.to(dt).to(DEV)
    got = []
    for rows in (wide.to(DEV)[:, :width], torch.where(wide == nan, 0, wide).to(DEV)):
        out = torch.empty(S, Hq, D, dtype=torch.bfloat16, device=DEV)
        ops.paged_attention_decode(out, q, kc, vc, rows, sl, starts, D ** -0.5, num_splits=nsplit, max_kv_len=700)
        got.append(out)
    assert not got[0].isnan().any() and torch.equal(got[0], got[1])


# (heads, key/value heads, values, page, e4m3, parts, sequences, most keys, tokens a sequence) and the checksum of the result's bytes
BITS = [((32, 8, 128, 16, False, 2, 25, 600, 1), 0xc6e13883),       # parts as waves of one workgroup
        ((32, 8, 128, 16, False, 1, 40, 1300, 1), 0x12719c80),
        ((32, 8, 128, 32, True, 1, 40, 1300, 1), 0x12dd8b1),
        ((16, 8, 64, 16, False, 7, 20, 3000, 1), 0xc8746bd1),
        ((16, 16, 64, 64, True, 2, 12, 500, 1), 0x9b88ecac),
        ((24, 8, 96, 16, False, 2, 30, 500, 4), 0x5dbefaa7),
        ((16, 8, 256, 16, False, 1, 30, 2000, 1), 0x102e32cf)]


@pytest.mark.parametrize("case,want", BITS)
def test_results_keep_their_bits(case, want):
    """The order in which products and the waves' sums are added is part of the result: a recorded run, replayed, gives its logits again.
    (Inputs are whole numbers over 64, the same wherever they are made.)"""
    Hq, Hkv, D, BS, fp8, parts, S, most, new = case
    lens = [max(new, 389 * (i + 1) % most) for i in range(S)]
    rng = np.random.RandomState(D + S)
    width = -(-max(lens) // BS)
    pages = len(lens) * width

    def some(*shape):
        return torch.from_numpy(rng.randint(-128, 129, shape).astype(np.float32) / 64).to(torch.bfloat16).to(DEV)

    q, k, v = some(len(lens) * new, Hq, D), some(pages, Hkv, BS, D), some(pages, Hkv, D, BS)
    table = torch.from_numpy(rng.permutation(pages).astype(np.int32)).view(len(lens), width).to(DEV)
    starts = torch.arange(len(lens) + 1, dtype=torch.int32, device=DEV) * new
    out = torch.empty_like(q)
    ops.paged_attention_decode(out, q, k.to(FP8) if fp8 else k, v.to(FP8) if fp8 else v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
                               starts, D ** -0.5, num_splits=parts, max_q_len=new)
    assert zlib.crc32(out.cpu().view(torch.uint8).numpy().tobytes()) == want
