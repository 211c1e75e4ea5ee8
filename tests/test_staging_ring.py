"""The pinned input buffers of graph replays (engine/graphs.StagingRing): a buffer is written again only behind an event that
covers its copy, on whichever streams the steps run."""
import random

import pytest
import torch

from distributed_llms_amd.engine import graphs


class _Stream:
    def __init__(self, handle, sid):
        self.handle, self.stream_id, self.issued, self.made = handle, sid, [], False

    @property
    def cuda_stream(self):                       # (torch makes a stream when its handle is first asked for)
        self.made = True
        return self.handle


class _Event:
    def __init__(self, log):
        self.log, self.covers = log, None

    def record(self, stream):
        self.covers = set(stream.issued)

    def synchronize(self):
        self.log |= self.covers


@pytest.mark.parametrize("ids", [(0, 3, 5, 8), (0, 4, 6, 9)])               # (whatever a stream's id says about its kind)
@pytest.mark.parametrize("seed", range(6))
def test_buffers_are_reused_behind_their_copies(monkeypatch, seed, ids):
    """Random walks over the default stream, two that the owner keeps and a caller's (never recorded on after its step)."""
    rng, done, events = random.Random(seed), set(), []
    streams = [_Stream(h, i) for h, i in zip((0, 11, 12, 13), ids)]
    now = [streams[seed % 3]]
    monkeypatch.setattr(graphs, "current_stream", lambda: now[0].cuda_stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: now[0])

    def event(stream):
        assert stream is now[0] or stream is not streams[3]
        e = _Event(done)
        e.record(stream)
        events.append(e)
        return e
    monkeypatch.setattr(graphs.StagingRing, "_event", staticmethod(event))
    ring, last = graphs.StagingRing(4), {}
    for s in streams[1:3]:
        ring.keep(s)
    used, steps = {now[0]}, 400
    for step in range(steps):
        if rng.random() < (0.0, 0.0, 0.1, 0.3, 0.9, 0.02)[seed]:
            now[0] = rng.choice(streams)
            used.add(now[0])
        buf = ring.take()
        assert buf not in last or last[buf] in done, (step, buf)
        last[buf] = step
        now[0].issued.append(step)
        ring.sent()
    assert {s for s in streams if s.made} == used
    if seed < 2:
        assert len(events) == steps // (ring.BUFFERS // 2)


@pytest.mark.gpu
def test_host_runs_ahead_of_replays(cuda):
    """Steps issued behind a long kernel, several times around the ring, each with inputs of its own: the outputs of steps that
    were waited for one by one."""
    from distributed_llms_amd.config import EngineConfig, get_model_config
    from distributed_llms_amd.engine.llm_engine import LLMEngine
    from distributed_llms_amd.engine.replay import TraceReplayer
    from distributed_llms_amd.models import weights as W
    from distributed_llms_amd.models.stage import ModelStage
    name = "tiny-llama-d128"
    cfg = get_model_config(name)
    stage = ModelStage(cfg, 0, cfg.num_layers, "cuda:0", torch.bfloat16).load_hf_state(W.synth_hf_state_dict(cfg, seed=1, dtype=torch.float32))
    eng = LLMEngine(EngineConfig(model=name, dtype="bfloat16", device="cuda", max_batch=2, max_seq_len=256, num_kv_blocks=64,
                                 graph_batch_sizes=(2,)), stage)
    steps, other = 3 * graphs.StagingRing.BUFFERS + 1, torch.cuda.Stream()
    assert eng.streams[0] in eng.runner.graphs.staging.kept

    def run(ahead):
        rp = TraceReplayer(eng)
        out = [rp.step([("a", [3, 5, 7], [2]), ("b", [2, 4], [1])])]
        torch.cuda.synchronize()
        if ahead:
            torch.cuda._sleep(200_000_000)
        for k in range(steps):
            if ahead == 2 and k in (5, 9):                       # a few steps in the middle on another stream
                other.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(other if ahead == 2 and 5 <= k < 9 else torch.cuda.current_stream()):
                out.append(rp.step([("a", [11 + k], [0]), ("b", [400 - 3 * k], [0])], end=("a", "b") if k == steps - 1 else ()))
            if ahead == 2 and k == 8:
                torch.cuda.current_stream().wait_stream(other)
            if not ahead:
                torch.cuda.synchronize()
        torch.cuda.synchronize()
        return out

    ref = run(0)
    for ahead in (1, 2):
        assert all(torch.equal(a, b) for a, b in zip(run(ahead), ref))
