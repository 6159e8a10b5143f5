"""The eager pass ahead of a capture runs after everything it reads."""

from __future__ import annotations

import contextlib

import torch


def test_first_pass_of_a_capture_waits_for_what_it_reads(monkeypatch):
    """The eager pass before a capture runs on a stream of its own: it has to wait
    for the stream that fills the static inputs."""
    from vllm_tgis_adapter_amd.engine.graph_runner import DecodeGraphRunner

    done = []

    class Stream:
        def __init__(self, name="side"):
            self.name = name

        def wait_stream(self, other):
            done.append(("wait", self.name, other.name))

    class Graph:
        def pool(self):
            return 0

    class Model:
        def __call__(self, ids, *_):
            done.append(("pass",))
            return ids

        def compute_logits(self, hidden):
            return hidden

    for name, f in [("Stream", Stream), ("CUDAGraph", Graph), ("synchronize", lambda: None),
                    ("stream", lambda s: contextlib.nullcontext()),
                    ("graph", lambda g, pool=None: contextlib.nullcontext()),
                    ("current_stream", lambda: Stream("current"))]:
        monkeypatch.setattr(torch.cuda, name, f)
    DecodeGraphRunner(Model(), [], None, 16, 2, 64, "cpu").capture()
    assert done.index(("wait", "side", "current")) < done.index(("pass",))


def test_a_packed_buffer_is_free_before_the_step(monkeypatch):
    """Its event stands behind the launch that reads it, not behind the whole replay."""
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.engine.graph_runner import DecodeGraphRunner

    done = []

    class Marks:
        def __init__(self, name):
            self.name = name

        def record(self):
            done.append(self.name)

        replay = record

    runner = DecodeGraphRunner(None, [], None, 16, 2, 64, "cpu")
    runner.graphs = {b: Marks("step") for b in runner.buckets}
    runner.out_logits = {b: torch.zeros(b, 1) for b in runner.buckets}
    monkeypatch.setattr(ops, "decode_inputs", lambda *_: done.append("read by"))
    runner.run_packed(torch.zeros(64, dtype=torch.uint8), 1, 1, Marks("event"))
    assert done == ["read by", "event", "step"]
