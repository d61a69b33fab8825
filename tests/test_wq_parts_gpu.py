"""Packed products at either side of the lines by which K is cut into parts (ops/csrc/gemm_wq.hip wq_parts): one part with a workgroup on most
CUs, as many parts as fit, one round of the two widths of workgroups.

Tolerance: as for the other packed products: fp32 sums of weights rounded to the activations' type, one rounding of the result (2^-8 of it in
bfloat16) and, as the 4-bit form scales its sums instead of the weights, one more of each product (2^-9, in quadrature): 2^-7 in norm is twice both."""
import pytest
import torch

from vllm_distributed_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K,rows", [(21888, 1024, (1, 16, 33, 64)), (28672, 2048, (2, 32, 33, 65)), (32896, 1024, (13, 64)), (10240, 8192, (13, 64, 65, 128)),
                                      (9216, 4096, (64, 65, 128)), (24448, 1024, (65, 128))])
def test_parts(bits, N, K, rows):
    g = torch.Generator(device=DEV).manual_seed(N + bits)
    group, most = 128, 15 if bits == 4 else 255
    q = torch.randint(0, most + 1, (N, K), generator=g, device=DEV, dtype=torch.uint8)
    scales = (torch.rand(N, K // group, generator=g, device=DEV) + 0.5).div_(most * K ** 0.5).bfloat16()
    zeros = torch.randint(most // 2, most // 2 + 2, (N, K // group), generator=g, device=DEV).bfloat16()
    sz = torch.stack([scales.t(), zeros.t()], -1).contiguous()
    qw = ops.w4_pack(q) if bits == 4 else q
    w = (q.float().view(N, -1, group) - zeros.float()[:, :, None]) * scales.float()[:, :, None]
    w = w.view(N, K)
    x = torch.randn(max(rows), K, generator=g, device=DEV).bfloat16()
    ref = x.double() @ w.double().t()
    for m in rows:
        got = ops.wq_gemm(x[:m], qw, sz, group, bits).double()
        assert float(((got - ref[:m]).norm(dim=1) / ref[:m].norm(dim=1)).max()) < 2 ** -7
