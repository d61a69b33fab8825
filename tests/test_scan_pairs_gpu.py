"""State-space kernels (ops/csrc/mamba.hip) at the edges of their forms against the token-by-token PyTorch form: channels in
pairs and odd ones, chunk and tile edges, groups that a workgroup's channels span, single tokens, padded rows."""
import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _scan_inputs(new, ctx, Ch, N, heads, groups, dtype, seed, offset=0):
    g = torch.Generator().manual_seed(seed)
    T, E = sum(new), heads or Ch

    def rows(width, std=1.0):                                       # ``offset`` values off a pair's boundary
        full = torch.randn(T, width + 2, generator=g) * std
        return full.to(dtype).to(DEV)[:, offset:offset + width]
    A = -(0.2 + torch.rand(E, generator=g)) if heads else -(0.2 + 2 * torch.rand(Ch, N, generator=g))
    S = len(new)
    return dict(u=rows(Ch), delta=rows(E, 0.5), A=A.to(DEV), B=rows(groups * N), C=rows(groups * N),
                D=torch.randn(E, generator=g).to(DEV), z=rows(Ch), delta_bias=(torch.randn(E, generator=g) - 2).to(DEV),
                ssm_state=torch.randn(S + 2, Ch, N, generator=g).to(DEV),
                query_start_loc=torch.tensor([0] + new).cumsum(0).int().to(DEV),
                seq_lens=torch.tensor([a + b if a + b else 0 for a, b in zip(new, ctx)]).int().to(DEV),
                block_table=(torch.randperm(S + 2, generator=g)[:S, None]).int().to(DEV), num_groups=groups)


@pytest.mark.parametrize("new,ctx", [([1, 1, 0, 1], [0, 5, 0, 9]),         # single tokens, a padded row
                                     ([31, 32, 33, 1, 0], [0, 3, 0, 4, 0]),
                                     ([95, 96, 97, 3], [7, 0, 1, 0]),       # chunked from 96 tokens on
                                     ([300, 64, 65], [0, 2, 0])])
@pytest.mark.parametrize("Ch,N,heads,groups", [(520, 16, 0, 1), (6, 16, 0, 1), (64, 16, 0, 4), (7, 16, 0, 1), (96, 32, 6, 1),
                                               (96, 64, 12, 2), (192, 128, 3, 1), (64, 256, 8, 1), (64, 128, 64, 1)])
def test_selective_scan_forms(new, ctx, Ch, N, heads, groups):
    a = _scan_inputs(new, ctx, Ch, N, heads, groups, torch.float32, Ch + N + len(new))
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, max_query_len=max(new))
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"], num_groups=groups)
    # 32-bit sums of N states, each carried through up to 300 decays below one
    torch.testing.assert_close(y, want, atol=3e-4, rtol=1e-4)
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("Ch,N,heads", [(1024, 16, 0), (256, 128, 4)])
def test_continued_sequences_of_many_chunks(Ch, N, heads):
    # the first chunk starts from the slot into which the last one leaves its state, here as soon as it has walked one token
    new, ctx = [97, 129, 161, 225, 257], [4, 1, 0, 9, 3]
    a = _scan_inputs(new, ctx, Ch, N, heads, 1, torch.float32, 11)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    first = a["ssm_state"].clone()
    ys = []
    for _ in range(3):
        a["ssm_state"].copy_(first)
        ys.append(ops.selective_scan(**a, max_query_len=max(new)))
        torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)
    torch.testing.assert_close(ys[0], want, atol=3e-4, rtol=1e-4)          # as in test_selective_scan_forms
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])


@pytest.mark.parametrize("Ch,N,heads,offset", [(520, 16, 0, 0), (96, 64, 12, 0), (7, 16, 0, 0), (64, 16, 0, 1)])
@pytest.mark.parametrize("new,ctx,hint", [([40, 3, 700], [0, 5, 2], None),          # the argument left out
                                          ([2, 0, 1, 0], [3, 4, 0, 0], None),       # ... and few rows: the one-token form
                                          ([900, 300], [1, 0], 128), ([900, 300], [1, 0], 256)])
def test_a_length_hint_that_is_too_small(new, ctx, hint, Ch, N, heads, offset):
    a = _scan_inputs(new, ctx, Ch, N, heads, 1, torch.float32, 5, offset)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, **({} if hint is None else dict(max_query_len=hint)))
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    torch.testing.assert_close(y, want, atol=3e-4, rtol=1e-4)              # as in test_selective_scan_forms
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


def test_rows_off_a_pair_boundary_take_the_plain_form():
    new, ctx = [130, 4], [0, 1]
    a = _scan_inputs(new, ctx, 64, 16, 0, 1, torch.bfloat16, 3, offset=1)
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, max_query_len=130)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    torch.testing.assert_close(y.float(), want.float(), atol=0.05, rtol=2 ** -7)      # one bf16 rounding of |y| below 8


@pytest.mark.parametrize("W", [2, 4, 8])
@pytest.mark.parametrize("C,offset", [(264, 0), (264, 1), (7, 0)])            # four channels a thread, or one
def test_conv_chunk_edges(W, C, offset):
    g = torch.Generator().manual_seed(W + C)
    new, ctx = [1, 2, 31, 32, 33, 70, 0], [0, 3, 0, 2, 1, 5, 0]
    x = torch.randn(sum(new), C + 4, generator=g).to(DEV)[:, offset:offset + C]
    w, b = torch.randn(C, W, generator=g).to(DEV), torch.randn(C, generator=g).to(DEV)
    state = torch.randn(9, C, W - 1, generator=g).to(DEV)
    qsl = torch.tensor([0] + new).cumsum(0).int().to(DEV)
    lens = torch.tensor([n + c for n, c in zip(new, ctx)]).int().to(DEV)
    table = torch.randperm(9, generator=g)[:7, None].int().to(DEV)
    st2 = state.clone()
    want = R.causal_conv1d(x, w, b, st2, qsl, lens, table)
    for longest in (max(new), 1, 9, 40):                                       # a hint only: results do not depend on it
        st = state.clone()
        y = ops.causal_conv1d(x, w, b, st, qsl, lens, table, longest)
        torch.testing.assert_close(y, want, atol=1e-5, rtol=1e-5)
        assert torch.equal(st, st2)


@pytest.mark.parametrize("Ch,repeat,form", [(520, 1, "vda_selective_scan"), (4104, 5, "vda_selective_scan_pairs")])
def test_short_sequences_take_the_form_that_fills_the_chip(monkeypatch, Ch, repeat, form):
    new, ctx = [31, 32, 33, 1, 0] * repeat, [0, 3, 0, 4, 0] * repeat
    a = _scan_inputs(new, ctx, Ch, 16, 0, 1, torch.float32, 2)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append(name), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=33)
    assert called == [form]
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    torch.testing.assert_close(y, want, atol=3e-4, rtol=1e-4)              # as in test_selective_scan_forms
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("Ch,N,heads,repeat,longest,form", [(1024, 128, 16, 3, 33, "vda_selective_scan"), (1024, 128, 16, 4, 33, "vda_selective_scan_pairs"),
                                                            (1024, 256, 16, 2, 33, "vda_selective_scan_pairs"), (1024, 128, 16, 1, 8, "vda_selective_scan"),
                                                            (1024, 128, 16, 2, 8, "vda_selective_scan_pairs"), (64, 64, 2, 1, 33, "vda_selective_scan_pairs")])
def test_wide_states_of_few_short_sequences(monkeypatch, Ch, N, heads, repeat, longest, form):
    """As above for 64, 128 and 256 states a channel, where lanes of 16 states count."""
    new, ctx = [longest - 2, longest - 1, longest, 1, 0] * repeat, [0, 3, 0, 4, 0] * repeat
    a = _scan_inputs(new, ctx, Ch, N, heads, 1, torch.float32, 3)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append(name), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=longest)
    assert called == [form]
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    # as in test_selective_scan_forms, with N / 16 as many terms in a sum
    torch.testing.assert_close(y, want, atol=3e-4 * (N // 16) ** 0.5, rtol=1e-4)
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("Ch,N,S", [(16, 16, 3), (70, 16, 2), (4096, 16, 79), (4096, 16, 80), (4096, 16, 81), (33, 128, 3), (2048, 64, 39), (2048, 64, 41),
                                    (66, 256, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_token_of_few_and_of_many_sequences(Ch, N, S, dtype):
    """Both splits of the one-token kernel, on either side of where they change (5 Mi states) and where channels end inside a wave."""
    new, ctx = [1] * S, [i % 3 for i in range(S)]
    a = _scan_inputs(new, ctx, Ch, N, 0 if N == 16 else 1 if Ch % 2 else 2, 1, dtype, 6)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, max_query_len=1)
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    tol = 3e-4 * max(N // 16, 1) ** 0.5
    if dtype == torch.float32:
        torch.testing.assert_close(y, want, atol=tol, rtol=1e-4)
    else:                                                                   # the reference sums in fp32 as well; one rounding each: 2^-8
        torch.testing.assert_close(y.float(), want.float(), atol=tol, rtol=2.0 ** -7)
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("setting,tokens,offset,chunked", [(None, 200, 1, False), (None, 256, 1, True), ("64", 80, 1, True),
                                                          ("64", 80, 0, True), ("512", 300, 0, False), ("512", 300, 1, False)])
def test_the_chunk_setting_holds_for_both_forms(monkeypatch, setting, tokens, offset, chunked):
    monkeypatch.delenv("VDA_SCAN_CHUNK_MIN_TOKENS", raising=False)
    if setting is not None:
        monkeypatch.setenv("VDA_SCAN_CHUNK_MIN_TOKENS", setting)
    a = _scan_inputs([tokens, 5], [0, 2], 64, 16, 0, 1, torch.float32, 4, offset)
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append((name, args[-5])), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=tokens)
    (name, nchunks), = called
    assert (nchunks > 1) == chunked, called
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"])
    torch.testing.assert_close(y, want, atol=3e-4, rtol=1e-4)              # as in test_selective_scan_forms
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("Ch,groups,offset", [(64, 1, 0), (64, 2, 0), (72, 1, 0), (36, 1, 1), (7, 1, 0), (260, 1, 2)])
@pytest.mark.parametrize("new,ctx", [([96, 1, 8, 9, 0], [0, 4, 0, 1, 0]),            # eight tokens at a time, tiles of 32
                                     ([31, 32, 33, 130], [2, 0, 1, 0]), ([64, 65, 97, 2], [0, 5, 0, 3])])
@pytest.mark.parametrize("chunks", [False, True])
def test_two_states_a_lane(monkeypatch, new, ctx, Ch, groups, offset, chunks):
    # channels that do not fill a workgroup, rows that are read one value at a time, chunks of one tile (the setting asks for them)
    if chunks:
        monkeypatch.setenv("VDA_SCAN_CHUNK_MIN_TOKENS", "96")
    a = _scan_inputs(new, ctx, Ch, 16, 0, groups, torch.float32, Ch + len(new), offset)
    if not offset:
        a = {k: v.contiguous() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append((name, args[27], args[29])), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=max(new))
    assert called == [("vda_selective_scan_pairs", 2, -(-max(new) // 32) if chunks else 1)]
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"], num_groups=groups)
    torch.testing.assert_close(y, want, atol=3e-4, rtol=1e-4)              # as in test_selective_scan_forms
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("N,heads", [(16, 0), (128, 1)])
@pytest.mark.parametrize("S", [2, 63, 64, 65])
def test_sequences_are_taken_by_length(S, N, heads):
    # lengths that repeat, rise and fall, an absent one; more of them than are put in order
    new = [(37 * i) % 50 + 1 for i in range(S)]
    new[S // 2] = 0
    new[-1] = 90
    a = _scan_inputs(new, [i % 3 if n else 0 for i, n in enumerate(new)], 128, N, heads and 2, 1, torch.float16, S + N)
    a = {k: v.contiguous() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    f = {k: v.float() if isinstance(v, torch.Tensor) and v.dtype == torch.float16 else v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, max_query_len=90)
    want = R.selective_scan(*(f[k] for k in names), f["query_start_loc"], f["seq_lens"], f["block_table"])
    # 32-bit sums of N states carried through up to 90 decays, one fp16 rounding of the result
    torch.testing.assert_close(y.float(), want, atol=1e-3, rtol=2 ** -10)
    torch.testing.assert_close(a["ssm_state"], f["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("left_out", ["z", "D", "delta_bias"])
def test_two_states_a_lane_without(left_out):
    a = _scan_inputs([100, 3], [0, 2], 64, 16, 0, 1, torch.bfloat16, 9)
    a[left_out] = None
    if left_out == "D":                                                    # step sizes as they are: none below zero
        a["delta"], a["delta_bias"] = a["delta"].abs(), a["delta_bias"].abs() * 0.1
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    y = ops.selective_scan(**a, softplus=False, max_query_len=100) if left_out == "D" else ops.selective_scan(**a, max_query_len=100)
    want = R.selective_scan(*(b[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"], softplus=left_out != "D")
    # one bf16 rounding of y
    torch.testing.assert_close(y.float(), want.float(), atol=0.05, rtol=2 ** -7)
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("Ch,N,heads,groups", [(128, 64, 4, 1), (64, 128, 4, 1), (256, 128, 4, 2), (64, 256, 2, 2), (32, 128, 1, 1)])
@pytest.mark.parametrize("new,ctx", [([100, 1, 8, 9, 0], [0, 4, 0, 1, 0]),           # eight tokens at a time, tiles of 16
                                     ([15, 16, 17, 130], [2, 0, 1, 0]), ([64, 65, 97, 2], [0, 5, 0, 3])])
@pytest.mark.parametrize("chunks", [False, True])
def test_eight_states_a_lane(monkeypatch, new, ctx, Ch, N, heads, groups, chunks):
    # heads of one workgroup's channels and of several workgroups', chunks of two tiles (the setting asks for them)
    if chunks:
        monkeypatch.setenv("VDA_SCAN_CHUNK_MIN_TOKENS", "96")
    a = _scan_inputs(new, ctx, Ch, N, heads, groups, torch.float16, Ch + N + len(new))
    a = {k: v.contiguous() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    names = ("u", "delta", "A", "B", "C", "D", "z", "delta_bias", "ssm_state")
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append((name, args[27], args[29])), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=max(new))
    (name, form, nchunks), = called
    assert (name, form) == ("vda_selective_scan_pairs", 3) and (nchunks > 1) == chunks
    f = {k: v.float() if isinstance(v, torch.Tensor) and v.dtype == torch.float16 else v for k, v in b.items()}
    want = R.selective_scan(*(f[k] for k in names), b["query_start_loc"], b["seq_lens"], b["block_table"], num_groups=groups)
    live = torch.cat([torch.full((n,), bool(n + c)) for n, c in zip(new, ctx)]).to(DEV)
    # 32-bit sums of N states carried through up to 130 decays, one fp16 rounding of the result
    torch.testing.assert_close(y.float()[live], want[live], atol=1e-3, rtol=2 ** -10)
    torch.testing.assert_close(a["ssm_state"], f["ssm_state"], atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("S,tokens,Ch,N,cut", [(1, 160, 2048, 64, True), (1, 150, 2048, 64, False), (1, 160, 2048, 128, True), (1, 150, 2048, 128, False),
                                               (3, 256, 1024, 128, True), (3, 200, 1024, 128, False), (1, 600, 4096, 128, True), (1, 500, 4096, 128, False),
                                               (1, 160, 2048, 256, True), (3, 767, 2048, 128, False), (3, 768, 2048, 128, True), (4, 700, 2048, 64, True), (8, 700, 2048, 64, False)])
def test_prompts_are_cut_where_the_chip_has_room(monkeypatch, S, tokens, Ch, N, cut):
    """Eight states a lane: the rule by states and tokens, and the same result either way."""
    monkeypatch.delenv("VDA_SCAN_CHUNK_MIN_TOKENS", raising=False)
    a = _scan_inputs([tokens] * S, [i % 2 for i in range(S)], Ch, N, Ch // 64, 1, torch.float16, Ch + N)
    a = {k: v.contiguous() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    b = {k: v.clone() if isinstance(v, torch.Tensor) else v for k, v in a.items()}
    called, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *args: (called.append((name, args[27], args[29])), call(name, *args))[1])
    y = ops.selective_scan(**a, max_query_len=tokens)
    (name, form, nchunks), = called
    assert (name, form) == ("vda_selective_scan_pairs", 3) and (nchunks > 1) is cut
    monkeypatch.setenv("VDA_SCAN_CHUNK_MIN_TOKENS", "100000" if cut else "32")
    other = ops.selective_scan(**b, max_query_len=tokens)
    # sums of N states in another order over some hundred decays below one, and one fp16 rounding each
    torch.testing.assert_close(y.float(), other.float(), atol=2e-3, rtol=2 ** -9)
    torch.testing.assert_close(a["ssm_state"], b["ssm_state"], atol=2e-4, rtol=2e-4)
