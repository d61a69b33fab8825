"""Latent attention over LDS-staged tiles (ops/csrc/mla_tile.hip): what the kernel's inline statements leave to its author, read from the
assembly that the repository's own flags give (compiled here, no GPU)."""
import os
import re
import subprocess

import pytest

from vllm_distributed_amd.ops import build

SOURCE = os.path.join(build.HERE, "csrc", "mla_tile.hip")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instructions of each kernel, by its template arguments; a label is an entry that ends in a colon."""
    out = str(tmp_path_factory.mktemp("asm") / "mla_tile.s")
    cmd = [build._hipcc(), *build.DEVICE_FLAGS, *build.EXTRA_FLAGS["mla_tile.hip"], "--cuda-device-only", "-S", SOURCE, "-o", out]
    done = subprocess.run(cmd, capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    found, body = {}, None
    for line in open(out):
        head = re.match(r"_Z15mla_tile_kernelI(DF16b|DF16_)Li(\d)ELb(\d)ELb(\d)E", line)
        text = line.split(";")[0].strip()
        if head and text.endswith(":"):
            body = found.setdefault((head[1], int(head[2]), head[3] == "1", head[4] == "1"), [])
        elif line.startswith(".Lfunc_end"):
            body = None
        elif body is not None and text and (not text.startswith(".") or text.endswith(":")):
            body.append(text)
    assert len(found) == 16
    return found


def _blocks(body):
    """Basic blocks of a kernel: their instructions, and which blocks may follow each."""
    blocks, names = [[]], {}
    for text in body:
        if text.endswith(":"):
            blocks.append([])
            names[text[:-1]] = len(blocks) - 1
            continue
        blocks[-1].append(text)
        if text.startswith(("s_branch", "s_cbranch", "s_endpgm")):
            blocks.append([])
    after = []
    for i, b in enumerate(blocks):
        last = b[-1].split() if b else [""]
        to = [names[last[1]]] if last[0].startswith(("s_branch", "s_cbranch")) else []
        if not last[0].startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            to.append(i + 1)
        after.append(to)
    return blocks, after


def _copies(text):
    return text.startswith("buffer_load") and text.endswith("lds")


def test_copies_have_landed_before_rows_take_their_place(kernels):
    """Copies from global memory to LDS of the last key steps fill tiles that nobody reads; result rows are staged over them.  On every way from a
    copy to an LDS write that no copy can follow (those of the rows) all vector memory is waited for, and then for the other waves."""
    for which, body in kernels.items():
        blocks, after = _blocks(body)
        leads = [any(map(_copies, b)) for b in blocks]                  # a copy can follow the block's start
        assert any(leads) is not which[3]                               # (e4m3 rows pass registers)
        for _ in blocks:
            leads = [f or any(leads[k] for k in to) for f, to in zip(leads, after)]
        # 2: copies in flight, 1: this wave's have landed, the others' perhaps not, 0: all have
        state, todo, rows = [0] * len(blocks), list(range(len(blocks))), 0
        while todo:
            i = todo.pop()
            now = state[i]
            for at, text in enumerate(blocks[i]):
                if _copies(text):
                    now = 2
                elif re.match(r"s_waitcnt vmcnt\(0\)", text):
                    now = min(now, 1)
                elif text == "s_barrier":
                    now = 0 if now < 2 else 2
                elif text.startswith("ds_write") and not any(leads[k] for k in after[i]) and not any(map(_copies, blocks[i][at:])):
                    rows += 1
                    assert now == 0, (which, text)
            for k in after[i]:
                if now > state[k]:
                    state[k] = now
                    todo.append(k)
        assert rows >= 16, which


def _in_the_key_loop(body):
    """Blocks with products that lead back to themselves."""
    blocks, after = _blocks(body)
    for i, b in enumerate(blocks):
        if not any(t.startswith("v_mfma") for t in b):
            continue
        seen, todo = set(), list(after[i])
        while todo:
            k = todo.pop()
            if k not in seen:
                seen.add(k)
                todo += after[k]
        if i in seen:
            yield b


def test_key_loop_fetches_nothing_from_scratch(kernels):
    """A register that comes back from scratch inside the key loop is waited for together with every copy issued before it."""
    for which, body in kernels.items():
        for b in _in_the_key_loop(body):
            assert not any(t.startswith("scratch_") for t in b), which


def test_key_loop_moves_no_sums(kernels):
    """The products that add to the sums are opaque statements: a sum that the compiler copied just before or after one would lack the waits that
    it places around its own products."""
    for which, body in kernels.items():
        for b in _in_the_key_loop(body):
            assert not any(t.startswith("v_accvgpr_") for t in b), which
