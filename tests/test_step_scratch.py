"""The key/value cache leaves room for what the recurrences allocate in a step."""
import types

import pytest
import torch

from aws_k8s_ansible_provisioner_amd.engine.model_runner import ModelRunner
from aws_k8s_ansible_provisioner_amd.models.config import get_config
from aws_k8s_ansible_provisioner_amd.models.mudepel import MudepelLM
from aws_k8s_ansible_provisioner_amd.models.sazepel import SazepelLM


@pytest.mark.parametrize("name,cls", [("sazepel-w2048", SazepelLM), ("mudepel-w2048", MudepelLM)])
def test_cache_size(name, cls, monkeypatch):
    cfg = get_config(name)
    model = types.SimpleNamespace(cfg=cfg, _parts=SazepelLM._parts, hq=16, hkv=4, D=128, ffn=5632,
                                  kv_block_bytes=lambda *a: 1 << 20)
    model.step_scratch_bytes = lambda rows, seqs: cls.step_scratch_bytes(model, rows, seqs)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (250 << 30, 288 << 30))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda *a: 10 << 30)
    ecfg = types.SimpleNamespace(kv_cache_dtype="auto", gpu_memory_utilization=0.9, kv_cache_max_gib=0)
    runner = types.SimpleNamespace(model=model, ecfg=ecfg, mcfg=types.SimpleNamespace(
        hidden_size=2048, vocab_size=50000, num_layers=16), bs=32, is_gpu=True, device="cuda:0",
        cap_tokens=16640, max_seqs=256, max_blocks=128)
    with_scratch = ModelRunner._derive_num_blocks(runner)
    del model.step_scratch_bytes
    without = ModelRunner._derive_num_blocks(runner)
    scratch = cls.step_scratch_bytes(model, 16640, 256) >> 20       # (blocks of 1 MiB)
    assert 150 < scratch < 1024 and abs(without - with_scratch - scratch) <= 1
