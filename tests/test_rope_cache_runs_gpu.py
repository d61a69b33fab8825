"""Rotary embedding + cache write of long batches (ops/csrc/rope_cache.hip rope_and_cache_runs_kernel) where it can go wrong:
runs that start and end anywhere in a page and in the batch, tokens without a slot, single tokens between prompts, a batch
that is no multiple of a workgroup's tokens, pages of 16 to 64, partial and interleaved rotation, an e4m3 cache.

Values are copied (16 bits) or rounded once (e4m3): the same bytes as the reference.  Rotated numbers: two products and a sum in
fp32 and one rounding, which a fused multiply-add may turn by one unit in the last place; their e4m3 form likewise."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"
FP8 = torch.float8_e4m3fn


def _slots(runs, BS, pages, g):
    """One run per (first position, tokens), each in pages of its own; tokens < 0: that many tokens without a slot."""
    order, used, out = torch.randperm(pages, generator=g).tolist(), 0, []
    for first, n in runs:
        if n < 0:
            out += [-1] * -n
            continue
        own = order[used:used + (first + n - 1) // BS + 1]
        used += len(own)
        out += [own[(first + i) // BS] * BS + (first + i) % BS for i in range(n)]
    return torch.tensor(out, dtype=torch.int64)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("runs,BS,Hq,Hkv,D,rot,neox,fp8", [
    ([(0, 2051)], 16, 4, 2, 128, 128, True, False),
    ([(5, 700), (31, 16), (16, 16), (0, 15), (7, 1), (9, 1), (15, 1290), (1, 17)], 16, 8, 1, 128, 128, True, False),
    ([(3, 640), (0, -5), (8, 800), (0, -1), (0, 700)], 32, 7, 1, 96, 96, True, False),
    ([(13, 2100)] + [(k * 7 % 64, 1) for k in range(40)], 64, 3, 3, 64, 32, False, True),
    ([(13, 1000), (2, 1100)], 16, 6, 2, 256, 256, False, False),
    ([(100, 2100)], 48, 2, 1, 80, 48, True, True),                  # a page no power of two, six lanes a head
    ([(4, 1500), (20, 700)], 24, 4, 2, 128, 128, True, False),      # pages that runs of 16 do not divide: the general form
])
def test_runs(dt, runs, BS, Hq, Hkv, D, rot, neox, fp8):
    g = torch.Generator().manual_seed(len(runs) + BS)
    pages = 4200 // BS + 100
    slots = _slots(runs, BS, pages, g)
    T = slots.numel()
    assert T >= 2048
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, generator=g).to(dt).to(DEV)
    cs = torch.randn(4096, rot, generator=g).to(DEV)
    pos = torch.randint(0, 4096, (T,), generator=g).to(DEV)
    slots = slots.to(DEV)
    ct = FP8 if fp8 else dt
    kc = torch.zeros(pages, Hkv, BS, D, device=DEV, dtype=ct)
    vc = torch.zeros(pages, Hkv, D, BS, device=DEV, dtype=ct)
    ks, vs = (0.5, 0.25) if fp8 else (1.0, 1.0)
    want = qkv.clone()
    q, k, v = want[:, :Hq * D], want[:, Hq * D:(Hq + Hkv) * D], want[:, (Hq + Hkv) * D:]
    ops.rope_and_cache(pos, qkv, cs, kc, vc, slots, rot, D, Hq, Hkv, neox, ks, vs)
    R.rotary_embedding(pos, q, k, cs, rot, D, neox)
    u = 2.0 ** (-7 if dt == torch.bfloat16 else -10)
    torch.testing.assert_close(qkv.float(), want.float(), rtol=u, atol=2e-6)
    # the caches against the rows that the call itself left in qkv: exact
    got = qkv[:, Hq * D:].reshape(T, 2, Hkv, D)
    kw, vw = torch.zeros_like(kc), torch.zeros_like(vc)
    R.reshape_and_cache(got[:, 0].contiguous(), got[:, 1].contiguous(), kw, vw, slots, ks, vs)
    assert torch.equal(kc.view(torch.uint8), kw.view(torch.uint8))
    assert torch.equal(vc.view(torch.uint8), vw.view(torch.uint8))


@pytest.mark.parametrize("dt,neox,fp8", [(torch.bfloat16, True, True), (torch.float16, True, False), (torch.float16, False, True)])
def test_both_forms_give_the_same_bits(dt, neox, fp8):
    """A prompt written in one call, and in portions that are below the long form's first size."""
    g = torch.Generator().manual_seed(5)
    T, BS, Hq, Hkv, D = 1500, 16, 6, 2, 128
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, generator=g).to(dt).to(DEV)
    cs = torch.randn(T, D, generator=g).to(DEV)
    pos, slots = torch.arange(T, device=DEV), torch.arange(T, device=DEV) + 5
    got = []
    for portion in (T, 500):
        x = qkv.clone()
        kc = torch.zeros(T // BS + 2, Hkv, BS, D, device=DEV, dtype=FP8 if fp8 else dt)
        vc = torch.zeros(T // BS + 2, Hkv, D, BS, device=DEV, dtype=FP8 if fp8 else dt)
        for a in range(0, T, portion):
            ops.rope_and_cache(pos[a:a + portion], x[a:a + portion], cs, kc, vc, slots[a:a + portion], D, D, Hq, Hkv, neox)
        got.append([t.view(torch.uint8) for t in (x, kc, vc)])
    for a, b in zip(*got):
        assert torch.equal(a, b)
