"""The bound on a prompt's keys that the attention layers hand to the kernel (it says into how many parts keys are cut): the longest
of the step's prompts, and not of the sequences that decode beside them."""
import pytest
import torch

from vllm_distributed_amd import LLM, SamplingParams, ops


def _tiny(tmp):
    import transformers as tf
    torch.manual_seed(0)
    cfg = tf.LlamaConfig(vocab_size=320, hidden_size=128, intermediate_size=256, num_hidden_layers=1, num_attention_heads=2,
                         num_key_value_heads=1, max_position_embeddings=512, head_dim=64)
    tf.LlamaForCausalLM(cfg).float().save_pretrained(tmp, safe_serialization=True)


@pytest.mark.parametrize("run_ahead", [False, True])
def test_short_prompt_beside_a_long_decode(tmp_path, monkeypatch, run_ahead):
    _tiny(str(tmp_path))
    llm = LLM(model=str(tmp_path), skip_tokenizer_init=True, dtype="float32", device="cpu", max_model_len=512, max_num_seqs=4,
              enable_prefix_caching=False, async_scheduling=run_ahead)
    seen, prefill = [], ops.paged_attention_prefill

    def record(out, q, k_cache, v_cache, block_table, seq_lens, q_start_loc, scale, **kw):
        seen.append((kw["max_kv_len"], int(seq_lens.max())))
        return prefill(out, q, k_cache, v_cache, block_table, seq_lens, q_start_loc, scale, **kw)
    monkeypatch.setattr(ops, "paged_attention_prefill", record)
    sp = SamplingParams(temperature=0, max_tokens=12, ignore_eos=True)
    engine = llm.llm_engine
    engine.add_request("long", {"prompt_token_ids": [5 + i % 300 for i in range(400)]}, sp)
    for _ in range(4):
        engine.step()
    engine.add_request("short", {"prompt_token_ids": [7] * 20}, sp)
    while engine.has_unfinished_requests():
        engine.step()
    llm.shutdown()
    assert {longest for _, longest in seen} == {400, 20}
    assert all(bound == longest for bound, longest in seen), seen
