"""Which calls of ops.linear may leave the library for a launch on their operands' memory (ops.skinny_gemm_wanted): everything that the
library's operation takes, and the kernel would not, stays with it.  The rule is host code; CPU tensors stand in for device ones."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from vllm_distributed_amd import ops


@pytest.fixture(autouse=True)
def _as_on_a_device(monkeypatch):
    monkeypatch.setattr(ops, "_dev", lambda x: True)


def _operands(M=4, N=512, K=1024):
    return torch.randn(M, K).bfloat16(), torch.randn(N, K).bfloat16(), torch.randn(N).bfloat16()


def test_plain_calls_are_taken():
    x, w, b = _operands()
    assert ops.skinny_gemm_wanted(x, w) and ops.skinny_gemm_wanted(x, w, b)
    assert ops.skinny_gemm_wanted(x, torch.nn.Parameter(w, requires_grad=False), torch.nn.Parameter(b, requires_grad=False))
    with torch.no_grad():
        assert ops.skinny_gemm_wanted(x, torch.nn.Parameter(w), torch.nn.Parameter(b))


def test_other_biases_devices_and_shapes():
    x, w, b = _operands()
    for bias in (b[:1], b[0], b[:1].expand(512), b[None], b.float(), b.to("meta")):     # the library broadcasts some of these
        assert not ops.skinny_gemm_wanted(x, w, bias)
    assert not ops.skinny_gemm_wanted(x, w.to("meta"), b) and not ops.skinny_gemm_wanted(x.to("meta"), w, b)
    assert not ops.skinny_gemm_wanted(x, w[0], None)


def test_gradients_in_either_direction():
    x, w, b = _operands()
    for k in range(3):
        args = [t.clone().requires_grad_(i == k) for i, t in enumerate((x, w, b))]
        assert not ops.skinny_gemm_wanted(*args)
    with torch.autograd.forward_ad.dual_level():
        assert not ops.skinny_gemm_wanted(torch.autograd.forward_ad.make_dual(x, x), w, b)


def test_transforms_tracing_modes_and_autocast():
    x, w, b = _operands()
    seen = []

    def f(x, w, b):
        seen.append(ops.skinny_gemm_wanted(x, w, b))
        return torch.nn.functional.linear(x, w, b)

    torch.vmap(f, (0, None, None))(x[None].repeat(3, 1, 1), w, b)
    torch.vmap(f, (None, 0, None))(x, w[None].repeat(3, 1, 1), b)
    torch.func.jvp(lambda x: f(x, w, b), (x,), (x,))
    torch.func.grad(lambda x: f(x, w, b).float().sum())(x)
    torch.jit.trace(f, (x, w, b), check_trace=False)
    with FakeTensorMode() as mode:
        fake = [mode.from_tensor(t) for t in (x, w, b)]
        f(*fake)
    seen.append(ops.skinny_gemm_wanted(*fake))
    with torch.autocast("cpu", dtype=torch.bfloat16):
        f(x, w, b)

    class Named(torch.Tensor):
        pass

    f(x.as_subclass(Named), w, b)
    f(x, w.as_subclass(Named), b)
    assert len(seen) >= 10 and not any(seen)
