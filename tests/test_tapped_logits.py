"""Tapped logits on their way to the host: the step's own rows through pinned memory, a row per request at most; any others (all positions
of a prompt, say, which may be gigabytes) as they come, and the same numbers either way."""
import numpy as np
import pytest
import torch

from vllm_distributed_amd.entrypoints.trace_replay import TraceReplayer


@pytest.mark.parametrize("device,dtype", [("cpu", "float32"), pytest.param("cuda", "bfloat16", marks=pytest.mark.gpu)])
def test_only_the_steps_own_rows_are_pinned(tmp_path, monkeypatch, device, dtype):
    import transformers as tf
    torch.manual_seed(0)
    cfg = tf.LlamaConfig(vocab_size=320, hidden_size=128, intermediate_size=256, num_hidden_layers=1, num_attention_heads=2,
                         num_key_value_heads=1, max_position_embeddings=512, head_dim=64)
    tf.LlamaForCausalLM(cfg).float().save_pretrained(str(tmp_path), safe_serialization=True)
    r = TraceReplayer(str(tmp_path), dtype, 256, max_live=2, device=device, enforce_eager=True)
    pinned, empty = [], torch.empty

    def record(*a, **kw):
        t = empty(*a, **kw)
        if t.dim() == 2 and t.shape[1] == 320 and kw.get("dtype") == torch.float32 and t.device.type == "cpu":
            pinned.append((t.shape[0], t.is_pinned()))
        return t
    monkeypatch.setattr(torch, "empty", record)
    p = [5 + i for i in range(20)]
    every = r.step([{"id": "a", "tokens": p, "want": list(range(20))}], ["a"])
    assert not any(pin for _, pin in pinned)
    last = r.step([{"id": "b", "tokens": p, "want": [19]}], ["b"])
    assert [n for n, _ in pinned] == [1] and pinned[0][1] == (device == "cuda")
    assert every.shape == (20, 320) and np.abs(every[19] - last[0]).max() <= (1e-5 if device == "cpu" else 2.0 ** -7) * np.abs(last).max()
    r.shutdown()
