"""Which rows a replayed decode step returns, and that they stay what they were when the next step runs."""
import pytest
import torch

from distributed_llms_amd.config import EngineConfig, get_model_config
from distributed_llms_amd.engine.llm_engine import LLMEngine
from distributed_llms_amd.engine.replay import TraceReplayer
from distributed_llms_amd.models import weights as W
from distributed_llms_amd.models.stage import ModelStage


@pytest.mark.parametrize("target", ["cpu", pytest.param("gpu", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("want", [[1, 1, 1], [1, 0, 1], [0, 0, 1], [1, 1, 0]])
def test_rows_of_a_decode_step(target, want):
    """All rows in order are copied without a gather, some of them gathered: the same rows either way."""
    dev = "cuda" if target == "gpu" else "cpu"
    cfg = get_model_config("tiny-llama")
    sd = W.synth_hf_state_dict(cfg, seed=5, dtype=torch.float32)
    dtype = torch.bfloat16 if dev == "cuda" else torch.float32
    prompts = [[5, 6, 7], [9, 3], [1, 2, 3, 4, 8]]

    def replay(want):
        ecfg = EngineConfig(model="tiny-llama", dtype=str(dtype)[6:], device=dev, max_batch=4, max_seq_len=64, num_kv_blocks=32)
        rp = TraceReplayer(LLMEngine(ecfg, ModelStage(cfg, 0, cfg.num_layers, dev, dtype).load_hf_state(sd)))
        rp.step([(str(i), p, []) for i, p in enumerate(prompts)])
        out = []
        for k in range(3):
            out.append(rp.step([(str(i), [11 + i + k], [0] * want[i]) for i in range(3)]))
        return [o.cpu() for o in out]

    full, some = replay([1, 1, 1]), replay(want)
    rows = [i for i in range(3) if want[i]]
    for a, b in zip(full, some):
        assert b.dtype == torch.float32 and torch.equal(a[rows], b)
    assert not torch.equal(full[0], full[1])
