"""16-bit linears of few rows and small weights (ops.linear -> vda_skinny_gemm, eight waves a workgroup): the edges of the rule, numbers of
K chunks that eight waves do not share evenly, and rows that are a view.

Tolerance: fp32 sums of K products of exact 16-bit factors, relative error at most K 2^-24 of the sum of their sizes, then one rounding
to 16 bits (u = 2^-9 or 2^-12 of the value); with random signs the sum of the sizes is about K^0.5 of the result's size, so
u + K^1.5 2^-24 < 1.1 u in norm over a row."""
import pytest
import torch

from vllm_distributed_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,bias,taken", [(1, 256, 512, False, True), (16, 4096, 4096, True, True), (17, 4096, 2048, False, True),
                                              (16, 8192, 2048, False, True), (32, 8192, 1024, True, True), (32, 512, 2048, False, True),
                                              (5, 272, 1152, True, True), (16, 304, 3968, False, True), (11, 2064, 640, True, True),
                                              (17, 4096, 2176, False, False), (33, 512, 512, False, False), (16, 4112, 2176, False, False),
                                              (16, 4096, 4224, False, False), (1, 264, 512, False, False), (0, 256, 512, False, False)])
def test_few_rows(monkeypatch, dt, M, N, K, bias, taken):
    g = torch.Generator().manual_seed(M * N + K)
    wide = torch.randn(max(M, 1), K + 24, generator=g).to(dt).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dt).to(DEV)
    b = torch.randn(N, generator=g).to(dt).to(DEV) if bias else None
    calls, call = [], ops.N.call
    monkeypatch.setattr(ops.N, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    for x in (wide[:M, :K].contiguous(), wide[:M, 16:16 + K]):
        calls.clear()
        y = ops.linear(x, w, b)
        assert ("vda_skinny_gemm" in calls) is taken
        ref = x.double() @ w.double().t() + (0 if b is None else b.double())
        u = 2.0 ** (-9 if dt == torch.bfloat16 else -12)
        assert y.shape == (M, N)
        if M:
            assert float(((y.double() - ref).norm(dim=1) / ref.norm(dim=1)).max()) < 1.1 * u
    x = wide[:M, 3:3 + K]                                # not on 16 bytes: the library's
    calls.clear()
    assert ops.linear(x, w, b).shape == (M, N) and "vda_skinny_gemm" not in calls
