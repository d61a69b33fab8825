"""Products whose K is cut keep the parts' fp32 sums in memory of the call's own: how much a call asks for (on the host), and that
calls of two streams and of two threads do not meet in it."""
import threading

import pytest
import torch

from vllm_distributed_amd import ops
from vllm_distributed_amd.ops import native as N

host = pytest.mark.skipif(not N.is_available(), reason="libvda_ops.so is not built")
MOST = 128 << 20


def _wq(M, N_, K, G, bits, most=MOST, splits=0, variant=0):
    return N.value("vda_wq_gemm_slabs", M, N_, K, G, bits, N_, most, splits, variant)


def _dense(M, N_, K, most=MOST, splits=0, batch=1, epi=0):
    return N.value("vda_dense_gemm_slabs", M, N_, K, N_, epi, 0, splits, 0, batch, most)


@host
@pytest.mark.parametrize("ask", [lambda **kw: _wq(160, 6144, 4096, 128, 4, **kw), lambda **kw: _wq(60, 8192, 28672, 128, 4, **kw), lambda **kw: _dense(64, 4096, 8192, **kw),
                                 lambda **kw: _dense(64, 1024, 8192, batch=4, **kw), lambda **kw: N.value("vda_decode_gemm_slabs", 64, 2048, 8192, 2048, kw.get("most", MOST)),
                                 lambda **kw: N.value("vda_cb4_slabs", 16, 4096, 8192, kw.get("most", MOST) // 4, 0)])
def test_no_more_than_the_bound(ask):
    n = ask()
    assert n > 1 and ask(most=0) == 0
    size = [ask(most=m) for m in (1, 4 << 20, 8 << 20, 1 << 40)]
    assert size == sorted(size) and size[0] == 0 and size[-1] >= n


@host
def test_what_is_not_cut_asks_for_nothing():
    assert _wq(13, 57344, 8192, 128, 4) == 0 and _wq(512, 57344, 8192, 128, 4) == 0
    assert _wq(160, 6144, 4096, 128, 4, splits=1) == 0 and _wq(160, 6144, 4096, 128, 4, splits=3) == 3
    assert _wq(160, 6146, 4096, 128, 4) == 0                   # rows of four that sums are read in
    assert _wq(160, 6144, 4100, 128, 4) == 0 and _wq(0, 6144, 4096, 128, 4) == 0 and _dense(0, 4096, 8192) == 0      # not taken at all
    assert _wq(9, 300, 96, 32, 4, splits=5, variant=1) == 2    # units of 64: two of them
    assert _dense(4096, 8192, 8192) == 0 and _dense(64, 4096, 8192, splits=1) == 0


def _products():
    g = torch.Generator(device="cuda").manual_seed(5)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(torch.bfloat16)

    K, N_ = 8192, 2048
    qw = torch.randint(-2 ** 31, 2 ** 31, (N_, K // 8), generator=g, device="cuda").to(torch.int32)
    sz = torch.rand(K // 128, N_, 2, generator=g, device="cuda").to(torch.bfloat16)
    w = normal(N_, K)
    xs = [normal(160, K) for _ in range(2)]
    return [lambda i: ops.wq_gemm(xs[i], qw, sz, 128, 4, splits=8, variant=1), lambda i: ops.wq_gemm(xs[i][:40], qw, sz, 128, 4, splits=8, variant=2),
            lambda i: ops.dense_gemm(xs[i], w, splits=8), lambda i: ops.decode_gemm(xs[i][:64], w),
            lambda i: ops.grouped_linear(torch.stack([xs[i][:16], xs[1 - i][:16]]), torch.stack([w, w]))]


@pytest.mark.gpu
@pytest.mark.parametrize("which", range(5))
def test_two_streams_at_once(which):
    product = _products()[which]
    want = [product(i) for i in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(product(i))
    torch.cuda.synchronize()
    assert all(torch.equal(y, want[i]) for i in range(2) for y in got[i])


@pytest.mark.gpu
@pytest.mark.parametrize("which", range(5))
def test_two_threads_on_one_stream(which):
    """Each thread's second launch may come behind the other's first."""
    product = _products()[which]
    want = [product(i) for i in range(2)]
    got = [[], []]

    def run(i):
        for _ in range(30):
            got[i].append(product(i))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(len(got[i]) == 30 and torch.equal(y, want[i]) for i in range(2) for y in got[i])
