"""ops.linear where a call of few rows may not become a launch on its operands' memory: the library's results, on the device."""
import pytest
import torch

from vllm_distributed_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_calls_that_stay_with_the_library():
    g = torch.Generator().manual_seed(0)
    x, w, b = (torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((4, 1024), (512, 1024), (512,)))
    lin = torch.nn.functional.linear
    assert torch.equal(ops.linear(x, w, b[:1]), lin(x, w, b[:1]))                  # one value for all columns
    xs, ws = torch.stack([x, -x, 2 * x]), torch.stack([w, 2 * w])
    assert torch.equal(torch.vmap(lambda a: ops.linear(a, w, b))(xs), torch.vmap(lambda a: lin(a, w, b))(xs))
    assert torch.equal(torch.vmap(lambda a: ops.linear(x, a, b))(ws), torch.vmap(lambda a: lin(x, a, b))(ws))
    for f in (ops.linear, lin):
        y, t = torch.func.jvp(lambda a: f(a, w, b), (x,), (x + 1,))
        assert t.shape == y.shape and float(t.float().norm()) > 0
    bias = b.clone().requires_grad_(True)
    ops.linear(x, w, bias).float().sum().backward()
    assert torch.equal(bias.grad, torch.full_like(b, 4))
    with pytest.raises(RuntimeError):
        ops.linear(x, w.cpu(), b)
    with torch.autocast("cuda", dtype=torch.float16):
        assert ops.linear(x, w, b).dtype == torch.float16
