"""Rows spread over several workgroups (ops/csrc/sampling.hip, vocabularies of 8192 entries and more) against the
draw written out in 64 bits: thresholds by sorting, noise from the published hash of (seed, token)."""
import numpy as np
import pytest
import torch

from vllm_distributed_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _words(seed: int, V: int) -> np.ndarray:
    with np.errstate(over="ignore"):
        x = np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + np.arange(V, dtype=np.uint64) + np.uint64(0x632BE59BD9B4E019)
        for mul in (0xff51afd7ed558ccd, 0xc4ceb9fe1a85ec53):
            x ^= x >> np.uint64(33)
            x *= np.uint64(mul)
        x ^= x >> np.uint64(33)
    return (x >> np.uint64(16)).astype(np.uint32)


def _noise(seed: int, V: int) -> np.ndarray:
    return -np.log(-np.log(((_words(seed, V) >> np.uint32(8)).astype(np.float64) + 0.5) / 16777216.0))


def _noise32(seed: int, V: int) -> np.ndarray:
    """The same of the 32-bit u that the kernels have: close to 1, where the largest noise comes from, its steps are up to 1 % of that noise's exponential."""
    u = ((_words(seed, V) >> np.uint32(8)).astype(np.float32) + np.float32(0.5)) * np.float32(2.0 ** -24)
    return -np.log(-np.log(np.minimum(u, np.float32(1 - 2.0 ** -24)).astype(np.float64)))


def _scores(row, temp, k, p, mp, seed, noise=_noise):
    """Noisy logits of the kept tokens, -inf elsewhere, and the same with one more token kept at the top-p edge (its
    weight may fall on either side: weights are rounded to 2^-32 and come from a 32-bit exponential)."""
    z = row.double().numpy() / temp
    keep = np.ones(len(z), bool)
    order = np.argsort(-z, kind="stable")
    if 0 < k < len(z):
        keep = z >= z[order[k - 1]]
    edge = keep.copy()
    if p < 1:
        w = np.where(keep, np.exp(z - z.max()), 0.0)
        zs = z[order]
        above = np.concatenate([[0.0], np.cumsum(w[order])])[np.searchsorted(-zs, -z)]      # weight of the larger ones
        tol = 1e-5 * w.sum()
        edge = keep & (above < p * w.sum() + tol)
        keep = keep & (above < p * w.sum() - tol)
        if not keep.any():
            keep = z == z.max()
    if mp > 0:
        keep, edge = keep & (z >= z.max() + np.log(mp) + 1e-5), edge & (z >= z.max() + np.log(mp) - 1e-5)
    g = z + noise(seed, len(z))
    return np.where(keep, g, -np.inf), np.where(edge, g, -np.inf)


# 8192: the shortest split row; 8193: rows that no 16-byte load may read; 50257: odd chunks; one row: most workgroups
@pytest.mark.parametrize("V,S", [(8192, 12), (8193, 12), (50257, 24), (128256, 1)])
@pytest.mark.parametrize("shape", ["model", "flat", "ties", "masked"])
def test_split_rows_draw_what_the_sorted_form_draws(V, S, shape):
    g = torch.Generator().manual_seed(V + S)
    x = torch.randn(S, V, generator=g) * (0.05 if shape == "flat" else 2.0)
    if shape == "model":
        x.scatter_add_(1, torch.randint(0, V, (S, 30), generator=g), torch.rand(S, 30, generator=g) * 10)
    elif shape == "ties":
        x = (x * 2).round() / 2             # thousands of equal logits: the list overflows, the row is done alone
    elif shape == "masked":                 # a grammar leaves seven tokens; top-k reaches into the others
        x[:, torch.randperm(V, generator=g)[7:]] = -float("inf")
    r = torch.arange(S)
    temp = 0.4 + torch.rand(S, generator=g)
    temp[r % 6 == 5] = 0.0
    k = torch.where(r % 2 == 1, torch.randint(1, 60, (S,), generator=g), 0).to(torch.int32)
    p = torch.where(r % 4 >= 2, 0.3 + 0.65 * torch.rand(S, generator=g), 1.0)
    mp = torch.where(r % 5 == 4, 0.02, 0.0)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    got = ops.sample(*(t.to(DEV) for t in (x, temp, k, p, mp, seeds))).cpu()
    for s in range(S):
        t = int(got[s])
        if temp[s] == 0:
            assert t == int(x[s].argmax())
            continue
        sure, may = _scores(x[s], float(temp[s]), int(k[s]), float(p[s]), float(mp[s]), int(seeds[s]))
        # 32-bit logits below 64 after the temperature (2^-18 of rounding) and two 32-bit logarithms of arguments at
        # least 2^-25, the inner one of values near 1: 2^-14 covers both
        assert may[t] >= sure.max() - 2.0 ** -14, (s, t, sure.argmax())


def test_split_rows_of_nothing_but_masked_tokens():
    x = torch.full((4, 9000), -float("inf"), device=DEV)
    k = torch.tensor([0, 5, 0, 5], dtype=torch.int32, device=DEV)
    p = torch.tensor([1.0, 1.0, 0.5, 0.5], device=DEV)
    assert ops.sample(x, None, k, p).tolist() == [0, 0, 0, 0]


# a row of 8191 is walked by one workgroup, the same row and a masked entry by several; more rows than one set of launches takes;
# counts beyond the list's length, with and without a fraction
@pytest.mark.parametrize("S,high", [(600, 60), (24, 8191)])
@pytest.mark.parametrize("shape", ["model", "ties", "masked", "infinite"])
def test_both_forms_draw_the_same(S, high, shape):
    g = torch.Generator().manual_seed(S + len(shape))
    V = 8191
    x = torch.randn(S, V, generator=g) * 2.0
    if shape == "ties":
        x = (x * 2).round() / 2
    elif shape == "masked":
        x[:, 100:] = torch.where(torch.rand(S, V - 100, generator=g) < 0.7, -float("inf"), x[:, 100:])
    elif shape == "infinite":
        x[::2, 5] = float("inf")
        x[::3, 9] = torch.finfo(torch.float32).min
    r = torch.arange(S)
    temp = 0.4 + torch.rand(S, generator=g)
    k = torch.where(r % 2 == 1, torch.randint(high // 2, high, (S,), generator=g), 0).to(torch.int32)
    p = torch.where(r % 4 >= 2, 0.3 + 0.69 * torch.rand(S, generator=g), 1.0)
    mp = torch.where(r % 5 == 4, 0.02, 0.0)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    args = [t.to(DEV) for t in (temp, k, p, mp, seeds)]
    wide = torch.cat([x, torch.full((S, 1), -float("inf"))], 1)
    assert torch.equal(ops.sample(wide.to(DEV), *args), ops.sample(x.to(DEV), *args))


@pytest.mark.parametrize("S,V,split", [(3, 24575, False), (3, 24576, True), (33, 40959, False), (33, 40960, True),
                                       (257, 65535, False), (257, 65536, True)])
def test_unfiltered_rows(S, V, split):
    """Draws without top-k and top-p are spread over workgroups from longer rows on; temperature, min-p and greedy rows."""
    assert (ops.N.lib().vda_sample_workspace(S, V, 0) > 0) == split and ops.N.lib().vda_sample_workspace(S, V, 1) > 0
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(S, V, generator=g) * 2.0).to(DEV)
    temp = (0.4 + torch.rand(S, generator=g)).masked_fill_(torch.arange(S) % 3 == 2, 0.0).to(DEV)
    mp = torch.where(torch.arange(S) % 5 == 4, 0.02, 0.0).to(DEV)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g).to(DEV)
    got = ops.sample(x, temp, None, None, mp, seeds)
    off = torch.ones(S, device=DEV)                                          # a top-p that filters nothing: the other form
    assert torch.equal(got, ops.sample(x, temp, None, off, mp, seeds))
    assert torch.equal(got[2::3], x[2::3].argmax(1))


@pytest.mark.parametrize("high", [250, 300, 520])
def test_lists_of_about_256_entries(high):
    """Collected entries around the number up to which they are ranked; beyond, the radix descent."""
    test_both_forms_draw_the_same(24, high, "model")


def test_shares_beyond_what_a_sum_holds():
    """One workgroup a row of 66001 entries, most of them the maximum: their weights are summed in two goes."""
    g = torch.Generator().manual_seed(3)
    S, V = 300, 66001
    x = torch.randn(S, V, generator=g) * 2.0
    x[:4] = 0.0
    x[:4, ::8] = -1.0 - torch.rand(4, 8251, generator=g)
    p = torch.where(torch.arange(S) % 3 == 2, 1.0, 0.3 + 0.69 * torch.rand(S, generator=g))
    k = torch.where(torch.arange(S) % 4 == 1, 50, 0).to(torch.int32)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    few = [t.to(DEV) for t in (x[:8], k[:8], p[:8], seeds[:8])]              # 17 workgroups a row
    got = ops.sample(x.to(DEV), None, k.to(DEV), p.to(DEV), None, seeds.to(DEV))
    assert torch.equal(got[:8], ops.sample(few[0], None, few[1], few[2], None, few[3]))
    assert all(float(x[s, int(got[s])]) == 0.0 for s in range(2))            # top-p below the maxima's share of 0.95


def test_hash_whose_upper_word_changes_along_a_row():
    """Seeds that put the carry into the upper word of the noise's hash inside the row, and at a share's edges."""
    V, inverse = 40000, pow(0x9E3779B97F4A7C15, -1, 2 ** 64)
    seeds = []
    for at in (0, 1, 2047, 2048, 20001, V - 1):                             # the first token with the next upper word
        base = (0x12345678 << 32) - at
        seed = (base - 0x632BE59BD9B4E019) * inverse % 2 ** 64
        seeds.append(seed - 2 ** 64 if seed >= 2 ** 63 else seed)
    x = torch.randn(len(seeds), V, generator=torch.Generator().manual_seed(1)) * 0.1
    for p in (1.0, 0.7):
        got = ops.sample(x.to(DEV), None, None, torch.full((len(seeds),), p, device=DEV), None, torch.tensor(seeds, device=DEV)).cpu()
        for s, seed in enumerate(seeds):
            sure, may = _scores(x[s], 1.0, 0, p, 0.0, seed % 2 ** 64)
            assert may[int(got[s])] >= sure.max() - 2.0 ** -14               # as above


@pytest.mark.parametrize("V", [8191, 8192, 50257])                       # one workgroup a row, several
def test_a_nan_logit_weighs_nothing(V):
    """It is neither part of the weight that top-p takes a share of nor drawn: the row draws as if it were masked."""
    g = torch.Generator().manual_seed(V)
    S = 64
    x = torch.randn(S, V, generator=g) * 2.0
    x.scatter_add_(1, torch.randint(0, V, (S, 5), generator=g), torch.rand(S, 5, generator=g) * 10)
    at = torch.randint(0, V, (S, 1), generator=g)
    nan, masked = x.scatter(1, at, float("nan")), x.scatter(1, at, -float("inf"))
    p = 0.2 + 0.6 * torch.rand(S, generator=g)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    args = [None, None, p.to(DEV), None, seeds.to(DEV)]
    assert torch.equal(ops.sample(nan.to(DEV), *args), ops.sample(masked.to(DEV), *args))
    args[2] = None
    assert torch.equal(ops.sample(nan.to(DEV), *args), ops.sample(masked.to(DEV), *args))
    kept, want = ops.topk_topp_mask(nan.to(DEV), None, p.to(DEV)), ops.topk_topp_mask(masked.to(DEV), None, p.to(DEV))
    assert torch.equal(torch.where(kept.isnan(), -float("inf"), kept), want)


@pytest.mark.parametrize("V", [8191, 8192, 50257])
def test_a_row_of_nothing_but_nan_gives_a_token(V):
    """Nothing wins such a row; what comes out indexes the next step's embedding all the same."""
    x = torch.full((4, V), float("nan"), device=DEV)
    x[3, 5:] = -float("inf")
    t = torch.tensor([0.0, 1.0, 0.7, 1.0], device=DEV)
    for k, p in ((None, None), (torch.tensor([0, 5, 0, 5], dtype=torch.int32, device=DEV), torch.tensor([1.0, 1.0, 0.5, 0.5], device=DEV))):
        got = ops.sample(x, t, k, p)
        assert bool(((got >= 0) & (got < V)).all()), got
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        got = ops.argmax(x[:3].to(dt))
        assert bool(((got >= 0) & (got < V)).all()), got


# (length, seed, token) whose hash is the largest word: the noise of a u that rounds to 1 would be infinite
@pytest.mark.parametrize("V,seed,token", [(8191, 764, 290), (8191, 2558, 5888), (128256, 137, 125767), (128256, 236, 25723)])
@pytest.mark.parametrize("k", [0, 201])
def test_the_largest_word_is_finite_noise(V, seed, token, k):
    assert _words(seed, V)[token] >> np.uint32(8) == 0xffffff
    g = torch.Generator().manual_seed(seed)
    x = torch.full((1, V), -100.0)
    high = torch.randperm(V, generator=g)[:201]
    x[0, high[high != token][:200]] = torch.randn(200, generator=g)
    x[0, token] = -40.0                        # finite noise is at most log(2^24) = 16.7 there and at least -log(log(2^25)) = -2.9 elsewhere
    got = ops.sample(x.to(DEV), None, torch.tensor([k], dtype=torch.int32, device=DEV) if k else None, None, None,
                     torch.tensor([seed], device=DEV))
    assert int(got) != token and float(x[0, int(got)]) > -10.0


# logits on the bins' edges, far from zero (2^23 bins of 1 / 128 are 65536), in steps wider than the bins that are kept, and a single one far above the
# others; fractions close to one, and lists around the number that is ranked at once
@pytest.mark.parametrize("shape", ["edges", "far", "beyond", "steep", "peak", "hot"])
def test_bins_cut_where_the_one_workgroup_form_does(shape):
    g = torch.Generator().manual_seed(len(shape))
    S, V = 48, 8191
    x = torch.randn(S, V, generator=g) * 2.0
    temp = 0.4 + torch.rand(S, generator=g)
    if shape == "edges":
        x, temp = (x * 128).round() / 128, torch.ones(S)
    elif shape == "far":
        x = x + torch.where(torch.arange(S) % 2 == 0, 65000.0, -2.0e5)[:, None]
    elif shape == "beyond":
        x = x * 60
    elif shape == "steep":
        temp = torch.where(torch.arange(S) % 2 == 0, 2e-4, 2e-5)         # scaled logits on either side of 2^23 bins
    elif shape == "peak":
        x[:, 77] = 90.0
    else:
        temp = torch.full((S,), 30.0)
    r = torch.arange(S)
    k = torch.where(r % 3 == 1, torch.randint(1, 1200, (S,), generator=g), 0).to(torch.int32)
    p = torch.where(r % 3 == 1, torch.where(r % 2 == 0, 1.0, 0.9), torch.where(r % 2 == 0, 1.0 - torch.rand(S, generator=g) * 1e-4,
                                                                                torch.rand(S, generator=g)))
    mp = torch.where(r % 5 == 4, 0.02, 0.0)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    args = [t.to(DEV) for t in (temp, k, p, mp, seeds)]
    wide = torch.cat([x, torch.full((S, 1), -float("inf"))], 1)
    assert torch.equal(ops.sample(wide.to(DEV), *args), ops.sample(x.to(DEV), *args))


# rows of nearly equal logits are cut on finer grids: each of them, its ends, shares on different ones, shares further apart than a grid's ring, masked
# and NaN entries among them
@pytest.mark.parametrize("V", [8191, 20000])
@pytest.mark.parametrize("shape", [4.0, 1.0, 0.2, 0.05, 0.01, 0.002, 1e-4, 1e-6, "offset", "edges", "apart", "ramp", "peak", "masked", "nan"])
def test_flat_rows_are_cut_where_the_sorted_form_does(V, shape):
    g = torch.Generator().manual_seed(V + len(str(shape)))
    S = 24
    x = torch.randn(S, V, generator=g) * (shape if isinstance(shape, float) else 0.01)
    if shape == "offset":
        x = x + torch.tensor([1000.0, -300.0, 40000.0, 15.9])[torch.arange(S) % 4, None]
    elif shape == "edges":
        x = (x * 2 ** 17).round() / 2 ** 17
    elif shape == "apart":
        x[:, V // 2:] -= torch.tensor([0.3, 1.0, 5.0, 40.0])[torch.arange(S) % 4, None]
    elif shape == "ramp":
        x = x.sort(dim=1).values
        x[::2] *= 30.0
    elif shape == "peak":
        x[:, 77] = 9.0
    elif shape == "masked":
        x[:, V // 3:] = torch.where(torch.rand(S, V - V // 3, generator=g) < 0.7, -float("inf"), x[:, V // 3:])
        x[:4, 4096:] = -float("inf")
    elif shape == "nan":
        x.scatter_(1, torch.randint(0, V, (S, 3), generator=g), float("nan"))
    r = torch.arange(S)
    k = torch.where(r % 3 == 1, torch.randint(1, 3000, (S,), generator=g), 0).to(torch.int32)
    p = torch.where(r % 3 == 1, torch.where(r % 2 == 0, 1.0, 0.9), 0.02 + 0.97 * torch.rand(S, generator=g))
    temp = 0.4 + torch.rand(S, generator=g)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    args = [t.to(DEV) for t in (temp, k, p, None, seeds) if t is not None]
    args.insert(3, None)
    got = ops.sample(x.to(DEV), *args)
    if V == 8191:                              # one workgroup a row, several with a masked entry more
        assert torch.equal(ops.sample(torch.cat([x, torch.full((S, 1), -float("inf"))], 1).to(DEV), *args), got)
    if shape == "nan":
        return
    for s in range(S):
        sure, may = _scores(x[s], float(temp[s]), int(k[s]), float(p[s]), 0.0, int(seeds[s]), _noise32)
        # as above; offsets to 1e5 after the temperature: 2^-7 of rounding
        assert may[int(got[s])] >= sure.max() - (2.0 ** -6 if shape == "offset" else 2.0 ** -14), s


@pytest.mark.parametrize("std", [2.0, 0.3, 0.04, 0.02, 0.005, 5e-4])
@pytest.mark.parametrize("V", [128256, 151936])
def test_flat_rows_collect_short_lists(V, std):
    """Rows of nearly equal logits stay with the workgroups that share them: what is collected at the cut fits the list (4096 entries), else one
    workgroup does the row's ten passes alone.  A grid has 400 entries a bin on average or some 190 bins between a row's ends, whichever are more
    entries; between a normal distribution's, some 9 std, the densest point has 0.4 * 9 times the average: 2900 entries a bin of 151936."""
    g = torch.Generator().manual_seed(V)
    S, per_row, at = 8, 2320, 1792 // 4        # bytes of a row's workspace (SplitRow), words before its counts of collected entries, one a workgroup
    x = torch.randn(S, V, generator=g) * std
    x[0, 5] = -float("inf")
    temp = torch.where(torch.arange(S) % 4 == 3, 50.0, 1.0)
    k = torch.where(torch.arange(S) % 2 == 1, torch.tensor([50, 20000, 64000, V - 9])[torch.arange(S) // 2], 0).to(torch.int32)
    p = torch.where(torch.arange(S) % 2 == 0, torch.tensor([0.9, 0.5, 0.98, 0.1])[torch.arange(S) // 2], 1.0)
    seeds = torch.randint(0, 2 ** 62, (S,), generator=g)
    xd, td, kd, pd, sd = (t.to(DEV) for t in (x, temp, k, p, seeds))
    n = ops.N.lib().vda_sample_workspace(S, V, 1)
    ws = torch.zeros(n, dtype=torch.uint8, device=DEV)
    out = torch.empty(S, dtype=torch.long, device=DEV)
    ops.N.call("vda_sample", xd.data_ptr(), out.data_ptr(), td.data_ptr(), kd.data_ptr(), pd.data_ptr(), None, sd.data_ptr(), S, V, V, ws.data_ptr(),
               n, ops.N.stream())
    collected = ws[:per_row * S].view(torch.int32).view(S, -1)[:, at:at + 64].long() & 0xffffffff
    assert int(collected.sum(1).max()) <= 4096, collected.sum(1)
    assert torch.equal(out, ops.sample(xd, td, kd, pd, None, sd))
    for s in range(S):
        sure, may = _scores(x[s], float(temp[s]), int(k[s]), float(p[s]), 0.0, int(seeds[s]), _noise32)
        assert may[int(out[s])] >= sure.max() - 2.0 ** -14, s
