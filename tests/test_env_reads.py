"""Switches are read from the environment at the moment of the read, whatever stands in os.environ's place."""
import os

from vllm_distributed_amd import envs


def test_reads_follow_the_environment(monkeypatch):
    monkeypatch.delenv("VDA_MOE_ROWS_FORM", raising=False)
    default = envs.VDA_MOE_ROWS_FORM
    monkeypatch.setenv("VDA_MOE_ROWS_FORM", "2")
    assert envs.VDA_MOE_ROWS_FORM == 2 and default != 2
    monkeypatch.setenv("VLLM_API_KEY", "schätze")
    assert envs.VLLM_API_KEY == "schätze"
    monkeypatch.delenv("VDA_MOE_ROWS_FORM")
    assert envs.VDA_MOE_ROWS_FORM == default
    monkeypatch.setattr(os, "environ", {"VDA_MOE_ROWS_FORM": "1"})
    assert envs.VDA_MOE_ROWS_FORM == 1 and envs.VLLM_API_KEY is None
