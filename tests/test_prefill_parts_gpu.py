"""Prompts of few query tiles, whose keys are cut into parts (ops/csrc/attention.hip key_part, vda_prefill_parts): every head size, parts
without keys, tiles that end inside a part, every option, rows of no sequence; and the tile search over more than 64 sequences.

Tolerance as for decode attention: a weight is rounded to 16 bits (unit u) under a sum that is not, the output once more, so that an
element moves by at most 2 u max|v|; fp32 sums and the bare exponential add a few 1e-6 of it (1e-5 here)."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
FP8 = torch.float8_e4m3fn


def _batch(new, prefix, Hq, Hkv, D, BS, dt, fp8=False, spare=0):
    g = torch.Generator().manual_seed(len(new) * D + sum(prefix))
    lens = [a + b for a, b in zip(new, prefix)]
    need = [max(1, -(-n // BS)) for n in lens]
    order, at = torch.randperm(sum(need) + 2, generator=g), 0
    table = torch.zeros(len(new), max(need), dtype=torch.int32)
    for s, n in enumerate(need):
        table[s, :n] = order[at:at + n].to(torch.int32)
        at += n
    k, v = torch.randn(order.numel(), Hkv, BS, D, generator=g), torch.randn(order.numel(), Hkv, D, BS, generator=g)
    kc, vc = ((k.to(DEV).to(FP8), v.to(DEV).to(FP8)) if fp8 else (k.to(dt).to(DEV), v.to(dt).to(DEV)))
    q = torch.randn(sum(new) + spare, Hq, D, generator=g).to(dt).to(DEV)
    starts = torch.tensor([0] + new).cumsum(0).to(torch.int32).to(DEV)
    return q, kc, vc, table.to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV), starts


def _parts(b, Hq, keys=0):
    q, kc, _, table, sl, _ = b
    return ops.N.lib().vda_prefill_parts(sl.shape[0], q.shape[0], Hq, kc.shape[1], q.shape[2], keys or table.shape[1] * kc.shape[2])


@pytest.mark.parametrize("D,Hq,Hkv,BS,fp8", [(64, 8, 2, 16, False), (64, 4, 4, 64, True), (96, 6, 2, 16, False), (128, 8, 1, 16, False),
                                             (128, 14, 2, 32, True), (192, 4, 1, 32, False), (256, 4, 2, 16, False)])
@pytest.mark.parametrize("new,prefix", [([17], [1500]), ([33, 1, 128], [0, 900, 511]), ([5, 40, 16], [1023, 31, 480])])
def test_parts(D, Hq, Hkv, BS, fp8, new, prefix):
    b = _batch(new, prefix, Hq, Hkv, D, BS, torch.bfloat16, fp8)
    q, kc, vc, table, sl, starts = b
    assert _parts(b, Hq) > 1
    ks, vs = (0.5, 0.25) if fp8 else (1.0, 1.0)
    out = torch.empty_like(q)
    ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, D ** -0.5, k_scale=ks, v_scale=vs)
    want = R.paged_attention(q.float(), kc.float() * ks, vc.float() * vs, table, sl, starts, D ** -0.5)
    assert float((out.float() - want).abs().max()) <= (2 * 2.0 ** -9 + 1e-5) * float((vc.float() * vs).abs().max())


@pytest.mark.parametrize("kw", [dict(window=700), dict(chunk=640), dict(softcap=5.0), dict(causal=False), dict(v_shift=1), "sink", "alibi", "bias"])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_options_in_parts(D, kw):
    """The same call in one part: asked for its log-sum-exps, which are not cut."""
    Hq, Hkv = 8, 2
    b = _batch([20, 70], [1000, 1300], Hq, Hkv, D, 16, torch.float16)
    q, kc, vc, table, sl, starts = b
    assert _parts(b, Hq) > 1
    if kw == "sink":
        kw = dict(sink=torch.linspace(-1, 4, Hq, device=DEV))
    elif kw == "alibi":
        kw = dict(alibi=torch.linspace(0.001, 0.1, Hq, device=DEV))
    elif kw == "bias":
        kw = dict(dist_bias=ops.padded_distance_rows(torch.linspace(1, -1, 90 * Hq, device=DEV).view(90, Hq)))
    if kw.get("v_shift"):
        vc = vc[:, :1].contiguous()
    one, parts = torch.empty_like(q), torch.empty_like(q)
    ops.paged_attention_prefill(one, q, kc, vc, table, sl, starts, D ** -0.5, return_lse=True, **kw)
    ops.paged_attention_prefill(parts, q, kc, vc, table, sl, starts, D ** -0.5, **kw)
    assert float((one.float() - parts.float()).abs().max()) <= (4 * 2.0 ** -12 + 2e-5) * float(vc.float().abs().max())


def test_rows_of_no_sequence_stay_as_they_are():
    b = _batch([9, 30], [800, 600], 8, 1, 128, 16, torch.bfloat16, spare=5)
    q, kc, vc, table, sl, starts = b
    assert _parts(b, 8) > 1
    out = torch.full_like(q, 7.0)
    ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, 128 ** -0.5)
    assert bool((out[39:] == 7.0).all()) and not bool((out[:39] == 7.0).all())
    few = torch.empty_like(q[:39])                       # a bound that leaves one part
    ops.paged_attention_prefill(few, q[:39], kc, vc, table, sl, starts, 128 ** -0.5, max_kv_len=64)
    assert float((few.float() - out[:39].float()).abs().max()) <= 4 * 2.0 ** -9 * float(vc.float().abs().max())


@pytest.mark.parametrize("S", [1, 63, 64, 65, 130, 200])
@pytest.mark.parametrize("D", [96, 128])
def test_tile_search(S, D):
    new = [(7 * i) % 23 if i % 5 else 40 for i in range(S)]
    b = _batch(new, [3 * i % 50 for i in range(S)], 4, 4, D, 16, torch.bfloat16)
    q, kc, vc, table, sl, starts = b
    out = torch.empty_like(q)
    ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, D ** -0.5)
    live = [s for s in range(S) if new[s]]
    n_live = torch.tensor([0] + [new[s] for s in live]).cumsum(0).to(torch.int32).to(DEV)
    want = R.paged_attention(q.float(), kc.float(), vc.float(), table[live], sl[live], n_live, D ** -0.5)
    assert float((out.float() - want).abs().max()) <= (2 * 2.0 ** -9 + 1e-5) * float(vc.float().abs().max())


@pytest.mark.parametrize("D", [96, 192, 256])
@pytest.mark.parametrize("Hq,Hkv", [(6, 2), (64, 1), (80, 1)])           # a head group as wide as a workgroup's columns, and wider
@pytest.mark.parametrize("kw", [dict(), dict(window=50), dict(causal=False)])
def test_heads_that_are_no_power_of_two_or_wide(D, Hq, Hkv, kw):
    """Tiles and key steps that end inside a workgroup, every page size's rows in LDS."""
    for BS in (16, 32, 64):
        b = _batch([3, 64, 130, 33], [0, 31, 5, 64], Hq, Hkv, D, BS, torch.float16)
        q, kc, vc, table, sl, starts = b
        out = torch.empty_like(q)
        out, lse = ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, D ** -0.5, return_lse=True, **kw)
        want, want_lse = R.paged_attention(q.float(), kc.float(), vc.float(), table, sl, starts, D ** -0.5, return_lse=True, **kw)
        assert float((out.float() - want).abs().max()) <= (2 * 2.0 ** -12 + 1e-5) * float(vc.float().abs().max())
        torch.testing.assert_close(lse, want_lse.float(), atol=1e-4, rtol=1e-5)


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 8, 2), (128, 8, 1), (192, 4, 2), (256, 80, 1)])      # (the last: heads past a workgroup's columns)
@pytest.mark.parametrize("where", ["query", "key", "last key"])
def test_nan_comes_out_of_parts(D, Hq, Hkv, where):
    """A row that is NaN in one part (see test_options_in_parts) is NaN where its keys are cut."""
    b = _batch([20, 70], [1000, 1300], Hq, Hkv, D, 16, torch.bfloat16)
    q, kc, vc, table, sl, starts = b
    assert _parts(b, Hq) > 1
    if where == "query":
        q[3, 1], q[50, 0] = float("nan"), float("nan")
    else:
        at = 600 if where == "key" else 1369                       # of the second sequence; the last one is the last row's alone
        kc[int(table[1, at // 16]), Hkv - 1, at % 16, 5] = float("nan")
    one, parts = torch.empty_like(q), torch.empty_like(q)
    ops.paged_attention_prefill(one, q, kc, vc, table, sl, starts, D ** -0.5, return_lse=True)
    ops.paged_attention_prefill(parts, q, kc, vc, table, sl, starts, D ** -0.5)
    assert bool(one.isnan().any()) and torch.equal(one.isnan(), parts.isnan())


@pytest.mark.parametrize("keys", [1, 31, 96, 97, 200])
@pytest.mark.parametrize("kw", [dict(), dict(causal=False), dict(softcap=5.0), "sink"])
def test_short_prompts_of_96_values(keys, kw):
    """The direct form up to 96 keys, by the table or by the bound; options that it does not have, and longer prompts, in the other."""
    if kw == "sink":
        kw = dict(sink=torch.linspace(-1, 4, 6, device=DEV))
    b = _batch([min(keys, 40), 1, keys], [keys - min(keys, 40), keys - 1, 0], 6, 2, 96, 16, torch.float16)
    q, kc, vc, table, sl, starts = b
    tall = torch.cat([table, table.new_zeros(3, 40)], 1)
    one, two, three = torch.empty_like(q), torch.empty_like(q), torch.empty_like(q)
    ops.paged_attention_prefill(one, q, kc, vc, table, sl, starts, 96 ** -0.5, **kw)
    ops.paged_attention_prefill(two, q, kc, vc, tall, sl, starts, 96 ** -0.5, max_kv_len=keys, **kw)
    assert torch.equal(one, two) or keys > 80                       # (tables are whole pages: 96 keys are six)
    ops.paged_attention_prefill(three, q, kc, vc, tall, sl, starts, 96 ** -0.5, max_kv_len=640, return_lse=True, **kw)
    bound = (4 * 2.0 ** -12 + 2e-5) * float(vc.float().abs().max())
    assert float((one.float() - three.float()).abs().max()) <= bound and float((two.float() - three.float()).abs().max()) <= bound
    if "sink" not in kw:
        want = R.paged_attention(q.float(), kc.float(), vc.float(), table, sl, starts, 96 ** -0.5, **kw)
        assert float((one.float() - want).abs().max()) <= (2 * 2.0 ** -12 + 1e-5) * float(vc.float().abs().max())


@pytest.mark.parametrize("kw", [dict(chunk=96), dict(v_shift=1), "sink", "bias", "alibi", dict(window=70, softcap=5.0)])
@pytest.mark.parametrize("D", [96, 192])
@pytest.mark.parametrize("prefix", [0, 700])                            # one part, and (the last five tokens) several
def test_options_of_heads_of_96_and_192_values(D, kw, prefix):
    """Against the decode kernel, where every new token is a sequence of its own."""
    Hq, Hkv = 8, 2
    new = [150, 5] if not prefix else [5]
    b = _batch(new, [prefix] * len(new), Hq, Hkv, D, 16, torch.float16)
    q, kc, vc, table, sl, starts = b
    if kw == "sink":
        kw = dict(sink=torch.linspace(-1, 4, Hq, device=DEV))
    elif kw == "alibi":
        kw = dict(alibi=torch.linspace(0.001, 0.1, Hq, device=DEV))
    elif kw == "bias":
        kw = dict(dist_bias=ops.padded_distance_rows(torch.linspace(1, -1, 90 * Hq, device=DEV).view(90, Hq)))
    if kw.get("v_shift"):
        vc = vc[:, :1].contiguous()
    out, rows = torch.empty_like(q), torch.empty_like(q)
    ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, D ** -0.5, **kw)
    own = torch.cat([torch.full((n,), s) for s, n in enumerate(new)]).to(DEV)
    lens = torch.cat([prefix + 1 + torch.arange(n) for n in new]).to(torch.int32).to(DEV)
    each = torch.arange(len(own) + 1, dtype=torch.int32, device=DEV)
    ops.paged_attention_decode(rows, q, kc, vc, table[own].contiguous(), lens, each, D ** -0.5, **kw)
    assert float((out.float() - rows.float()).abs().max()) <= (4 * 2.0 ** -12 + 2e-5) * float(vc.float().abs().max())   # as above


@pytest.mark.parametrize("new", [[845], [846], [864], [430, 400], [500, 1, 700], [300] * 4])           # 47, 48, 49 tiles, and more of several prompts
def test_four_groups_of_tiles(new):
    """Four kv heads, whose tiles go to the XCDs in turn from 48 on and for up to three prompts, in runs otherwise: all of them, once each."""
    b = _batch(new, [5] * len(new), 28, 4, 128, 16, torch.bfloat16)
    q, kc, vc, table, sl, starts = b
    out = torch.full_like(q, float("nan"))
    ops.paged_attention_prefill(out, q, kc, vc, table, sl, starts, 128 ** -0.5, max_kv_len=32 * 15)      # (one part)
    want = R.paged_attention(q.float(), kc.float(), vc.float(), table, sl, starts, 128 ** -0.5)
    assert float((out.float() - want).abs().max()) <= (2 * 2.0 ** -9 + 1e-5) * float(vc.float().abs().max())
