"""A captured step's inputs from one packed host buffer (decode_inputs.hip): the same static
buffers as by copies, padding rows and tables' ends too, also when the buffer is written anew."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("states", [False, True])
@pytest.mark.parametrize(("n", "w", "rows", "blocks"), [
    (1, 1, 1, 1), (1, 15, 1, 512), (3, 0, 4, 7), (5, 300, 8, 300), (64, 257, 64, 600), (33, 2, 48, 3)])
def test_inputs(n, w, rows, blocks, states):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops
    from vllm_tgis_adapter_amd.engine.graph_runner import DecodeGraphRunner

    need = DecodeGraphRunner.packed_bytes(n, w)
    packed = torch.empty(need + 16, dtype=torch.uint8, pin_memory=True)
    host = packed.numpy()
    dev = dict(device="cuda")
    for seed in range(3):
        rng = np.random.default_rng(seed)
        longs = rng.integers(-1, 1 << 40, (3, n))
        ints = rng.integers(-1, 1 << 30, 2 * n).astype(np.int32)
        table = rng.integers(0, 1 << 30, (n, w)).astype(np.int32)
        host[:24 * n].view(np.int64).reshape(3, n)[:] = longs
        host[24 * n:32 * n].view(np.int32)[:] = ints
        host[32 * n:need].view(np.int32).reshape(n, w)[:] = table
        ids, pos, slots = (torch.full((rows + 1,), 77, dtype=torch.long, **dev) for _ in range(3))
        lens, st = (torch.full((rows + 1,), 77, dtype=torch.int32, **dev) for _ in range(2))
        tables = torch.full((rows + 1, blocks), 77, dtype=torch.int32, **dev)
        ops.decode_inputs(packed, ids, pos, slots, lens, st if states else None, tables, n, w, rows)
        torch.cuda.synchronize()

        def rest(values, pad, total=rows):
            return list(values) + [pad] * (total - n) + [77]

        assert ids.tolist() == rest(longs[0], 77)
        assert pos.tolist() == rest(longs[1], 77)
        assert slots.tolist() == rest(longs[2], -1)
        assert lens.tolist() == rest(ints[:n], 0)
        assert st.tolist() == (rest(ints[n:], -1) if states else [77] * (rows + 1))
        want = torch.full((rows + 1, blocks), 77, dtype=torch.int32)
        want[:n] = 0
        want[:n, :w] = torch.from_numpy(table)
        assert torch.equal(tables.cpu(), want)


def test_what_is_refused():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from vllm_tgis_adapter_amd import ops

    def call(n=2, w=3, rows=2, size=88, pinned=True, blocks=4):
        longs = [torch.zeros(2, dtype=torch.long, device="cuda") for _ in range(3)]
        ops.decode_inputs(torch.zeros(size, dtype=torch.uint8, pin_memory=pinned), *longs,
                          torch.zeros(2, dtype=torch.int32, device="cuda"), None,
                          torch.zeros((2, blocks), dtype=torch.int32, device="cuda"), n, w, rows)

    call()
    for bad in (dict(rows=3), dict(n=3), dict(size=87), dict(pinned=False), dict(blocks=2)):
        with pytest.raises(RuntimeError):
            call(**bad)
