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
