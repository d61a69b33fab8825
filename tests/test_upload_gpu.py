"""A step's host arrays in one launch (ops.upload, ModelRunner._queue_upload): every byte is where a copy would have put it and no other
byte changes."""
import numpy as np
import pytest
import torch

from vllm_distributed_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("sizes", [[(1, 1)], [(1, 3), (1, 4), (5, 7), (1, 65536), (3, 1)], [(12, 25)] * 16, [(2, k + 1) for k in range(19)]])
def test_blocks(sizes):
    host = torch.empty(1 << 20, dtype=torch.uint8).pin_memory()
    at, view = ops.mapped_host(host), host.numpy()
    g, off, blocks, want = np.random.default_rng(1), 0, [], []
    for k, (rows, width) in enumerate(sizes):
        src = g.integers(-2 ** 31, 2 ** 31, (rows, width), dtype=np.int32)
        view[off:off + src.nbytes].view(np.int32)[...] = src.reshape(-1)
        dst = torch.full((rows + 1, width + 3), -7, dtype=torch.int32, device=DEV)
        first = k % 4                                   # any alignment of four bytes
        blocks.append((at + off, dst.data_ptr() + 4 * first, width, rows, width + 3 if rows > 1 else 0))
        ref = torch.full((rows + 1, width + 3), -7, dtype=torch.int32)
        flat = ref.view(-1)
        for r in range(rows):
            flat[first + r * (width + 3):first + r * (width + 3) + width] = torch.from_numpy(src[r])
        want.append((dst, ref))
        off += (src.nbytes + 15) // 16 * 16 if k % 2 else src.nbytes
    ops.upload(blocks)
    for dst, ref in want:
        assert torch.equal(dst.cpu(), ref)


def test_nothing_and_refused():
    ops.upload([])
    d = torch.zeros(4, dtype=torch.int32, device=DEV)
    for bad in ((0, d.data_ptr(), 1, 1, 0), (d.data_ptr(), 0, 1, 1, 0), (d.data_ptr(), d.data_ptr() + 2, 1, 1, 0),
                (d.data_ptr(), d.data_ptr(), 0, 1, 0), (d.data_ptr(), d.data_ptr(), 2, 2, 1)):
        with pytest.raises(RuntimeError):
            ops.upload([bad])
    assert ops.mapped_host(torch.empty(16)) is None


def test_runner_queue_equals_copies():
    """The same arrays, queued and copied: other types are converted, what does not fit is left to the copy."""
    from vllm_distributed_amd.worker.model_runner import ModelRunner
    r = object.__new__(ModelRunner)
    r.is_gpu = r.pin = True
    r._stage_bufs, r._stage_idx, r._stage_off, r._stage_bytes, r._uploads = None, 0, 0, 1 << 19, None
    g = np.random.default_rng(2)
    arrays = [(torch.int32, g.integers(0, 9, 5)), (torch.int64, g.integers(0, 2 ** 40, 33)), (torch.float32, g.random(7)),
              (torch.int32, g.integers(0, 99, 70000).astype(np.int32)), (torch.int32, np.zeros(0, dtype=np.int32))]
    table = g.integers(0, 99, (6, 11)).astype(np.int32)
    got = []
    for queue in (False, True):
        r._stage_idx, r._stage_off = int(queue), 0
        dst = [torch.full((len(a) + 5,), 3, dtype=t, device=DEV) for t, a in arrays]
        tab = torch.full((9, 20), -1, dtype=torch.int32, device=DEV)
        if queue:
            r._start_uploads()
            assert r._uploads == []
        for d, (_, a) in zip(dst, arrays):
            r._to_dev(d, a)
        r._table_to_dev(tab, table)
        assert len(r._uploads or []) == (4 if queue else 0)      # (the largest goes by itself, the empty one nowhere)
        r._flush_uploads()
        assert r._uploads is None
        got.append([x.cpu() for x in dst + [tab]])
    for a, b in zip(*got):
        assert torch.equal(a, b)
