"""Multi-LoRA runtime.

Hot-loads PEFT LoRA adapters (adapter_config.json + adapter_model.safetensors)
onto the serving model and applies them per request in mixed batches.

Application model: each step batch carries a per-token adapter id; for every
active adapter the delta  x @ A^T @ B^T * (alpha/r)  is added onto the
matching projection outputs: on a GPU by the batched kernels of
kernels/lora_bgmv.hip over stacks of the active adapters, else grouped by
adapter.

TP sharding follows the base layer: column-parallel projections
(q/k/v/gate/up) shard B on the output dim; row-parallel projections (o/down)
shard A on the input dim.
"""

from __future__ import annotations

import json
import os
from dataclasses import dataclass, field
from typing import Optional

import torch

from .. import ops
from ..parallel import get_tp_rank, get_tp_world_size

# projection name -> (parallel kind, hf targets)
_COLUMN = {"q_proj", "k_proj", "v_proj", "gate_proj", "up_proj"}
_ROW = {"o_proj", "down_proj"}
_SUPPORTED = _COLUMN | _ROW


@dataclass
class LoRAAdapter:
    lora_int_id: int
    rank: int
    scaling: float
    # (layer_idx, proj) -> (A [r, in_local], B [out_local, r])
    weights: dict[tuple[int, str], tuple[torch.Tensor, torch.Tensor]]


@dataclass
class LoRAContext:
    """Per-step batch context set by the worker before the forward."""

    token_lora_ids: Optional[torch.Tensor] = None  # [T] int32 device (0 = none)
    adapters: dict[int, LoRAAdapter] = field(default_factory=dict)
    # BGMV kernel context (GPU): slot per token (-1 = none) + slot order
    token_slots: Optional[torch.Tensor] = None  # [T] int32 device
    slot_ids: tuple[int, ...] = ()

    @property
    def active(self) -> bool:
        return self.token_lora_ids is not None and bool(self.adapters)


CTX = LoRAContext()

# (slot_ids, layer, projections, dtype) -> (a_stack, b_stack, scales, spans)
_STACK_CACHE: dict = {}


def invalidate_adapter(lora_int_id: int) -> None:
    """Drop cached stacks containing this adapter (removal / reload)."""
    for key in [k for k in _STACK_CACHE if lora_int_id in k[0]]:
        del _STACK_CACHE[key]


_RECENT_SETS: list = []  # LRU of active-adapter sets whose stacks stay cached
_MAX_CACHED_SETS = 4


def set_context(token_lora_ids: Optional[torch.Tensor], adapters: dict[int, LoRAAdapter]) -> None:
    CTX.token_lora_ids = token_lora_ids
    CTX.adapters = adapters
    new_slot_ids = tuple(sorted(adapters))
    if new_slot_ids != CTX.slot_ids and adapters:
        # keep stacks for a small LRU of adapter sets (batches often
        # alternate between a few combinations); evict the rest so GPU
        # memory stays bounded
        if new_slot_ids in _RECENT_SETS:
            _RECENT_SETS.remove(new_slot_ids)
        _RECENT_SETS.append(new_slot_ids)
        if len(_RECENT_SETS) > _MAX_CACHED_SETS:
            _RECENT_SETS.pop(0)
            keep = set(_RECENT_SETS)
            for key in [k for k in _STACK_CACHE if k[0] not in keep]:
                del _STACK_CACHE[key]
    CTX.slot_ids = new_slot_ids
    CTX.token_slots = None
    if token_lora_ids is not None and adapters:
        CTX.token_slots = ops.lora_slots(token_lora_ids, CTX.slot_ids)


def clear_context() -> None:
    CTX.token_lora_ids = None
    CTX.adapters = {}
    CTX.token_slots = None
    CTX.slot_ids = ()


def _get_stacks(layer_idx: int, projs: list[tuple[str, int, int]], in_size: int,
                dtype: torch.dtype, device) -> Optional[tuple]:
    """Stacked, rank-padded (A, B, scales, spans) of the active adapter set for the
    projections of one input: A [L, P * R, in_size], B [L, V, R] (the projections'
    columns one after the other) and their spans of the output.  Projections that no
    adapter has are left out; None when that leaves none."""
    key = (CTX.slot_ids, layer_idx, tuple(projs), dtype)
    if key in _STACK_CACHE:
        return _STACK_CACHE[key]
    adapters = [CTX.adapters[lid] for lid in CTX.slot_ids]
    have = [(name, lo, hi) for name, lo, hi in projs
            if any((layer_idx, name) in a.weights for a in adapters)]
    if not have:
        _STACK_CACHE[key] = None
        return None
    rank = max(a.weights[(layer_idx, name)][0].shape[0]
               for a in adapters for name, _, _ in have if (layer_idx, name) in a.weights)
    rank = next((r for r in ops.LORA_RANKS if r >= rank), rank)
    L, width = len(adapters), sum(hi - lo for _, lo, hi in have)
    a_stack = torch.zeros((L, len(have) * rank, in_size), dtype=dtype, device=device)
    b_stack = torch.zeros((L, width, rank), dtype=dtype, device=device)
    scales = torch.tensor([ad.scaling for ad in adapters], dtype=torch.float32, device=device)
    for s, ad in enumerate(adapters):
        v = 0
        for p, (name, lo, hi) in enumerate(have):
            ab = ad.weights.get((layer_idx, name))
            if ab is not None:
                a, b = ab
                a_stack[s, p * rank: p * rank + a.shape[0]] = a
                b_stack[s, v: v + hi - lo, : b.shape[1]] = b
            v += hi - lo
    _STACK_CACHE[key] = (a_stack, b_stack, scales, [(lo, hi) for _, lo, hi in have])
    return _STACK_CACHE[key]


def _batched(x: torch.Tensor) -> bool:
    """Whether the batched kernels take the deltas of this input."""
    return (
        CTX.token_slots is not None
        and ops.native_enabled(x)
        and x.is_contiguous()
        and x.shape[1] % 8 == 0
        and all(a.rank <= 64 for a in CTX.adapters.values())
    )


# Most tokens, times a layer's 256-column pieces, up to which the gate is taken in the launch that
# adds the deltas, by rank (us there | deltas and gate apart; tokens x columns, 4 adapters): rank 8, 1024 x
# 16384 41 | 43, 2048 x 28672 104 | 113, 4096 x 28672 198 | 217; 16, 301 x 28672 26.7 | 27.3, 700 x 16384
# 36.0 | 36.2, 1000 x 28672 61.1 | 60.8; 32, 33 x 28672 13.9 | 15.3, 36 x 28672 15.1 | 16.3; past the line 61 x
# 28672 15.3 | 16.0, 512 x 28672 42 | 41, 1024 x 28672 74 | 75; 64, 16 x 16384 15.1 | 15.9; past the line,
# where the gate would be a column a thread, 16 x 28672 22.4 | 20.2, 512 x 28672 413 | 54.
_GATE_TILES = {8: 131072, 16: 32768, 32: 4096, 64: 1024}


def gate_with_deltas(tokens: int, width: int, rank: int) -> bool:
    """Whether the launch that adds the deltas to a gate and up product takes the gate too."""
    return tokens * ((width + 255) // 256) <= _GATE_TILES.get(rank, 0)


def lora_linear(
    layer_idx: int,
    projs: list[tuple[str, int, int]],
    x: torch.Tensor,
    weight: Optional[torch.Tensor],  # of the base linear, without a bias; None: not as it is
    base,                            # () -> its product
    gated: bool = False,
) -> Optional[torch.Tensor]:
    """The base linear's product with the adapters' deltas, made together where that is
    faster, gated: silu of the first half of its columns times the second.  None where the
    batched bf16 kernels do not apply: the caller has the product made, then apply_lora."""
    if not (CTX.active and x.dim() == 2 and x.dtype == torch.bfloat16 and len(projs) <= 3
            and _batched(x)):
        return None
    stacks = _get_stacks(layer_idx, projs, x.shape[1], x.dtype, x.device)
    if stacks is None:
        return None
    a_stack, b_stack, scales, spans = stacks
    slots = CTX.token_slots
    gate = False
    if gated:
        width = projs[-1][2]
        gate = gate_with_deltas(x.shape[0], width, b_stack.shape[2])
    out = None
    if weight is not None:
        out = ops.lora_product(x, weight, None, a_stack, b_stack, slots, scales, spans, gate)
    if out is None:
        y = base()
        if gate:
            out = ops.lora_product(x, None, y, a_stack, b_stack, slots, scales, spans, True)
        if out is None:
            gate = False
            if y.is_contiguous():
                ops.lora_delta(y, x, a_stack, b_stack, slots, scales, spans)
                out = y
            else:
                out = apply_lora(layer_idx, projs, x, y)
    return ops.silu_and_mul(out) if gated and not gate else out


def apply_lora(
    layer_idx: int,
    projs: list[tuple[str, int, int]],  # (proj name, out-slice start, out-slice end)
    x: torch.Tensor,     # [T, in_local] input of the base linear
    out: torch.Tensor,   # [T, sum(out_local)] output to update in place
) -> torch.Tensor:
    if not CTX.active:
        return out
    # GPU: batched BGMV shrink/expand HIP kernels over the mixed batch (E12)
    if _batched(x) and out.is_contiguous():
        if x.dtype == torch.bfloat16 and len(projs) <= 3:
            stacks = _get_stacks(layer_idx, projs, x.shape[1], x.dtype, x.device)
            if stacks is not None:
                a_stack, b_stack, scales, spans = stacks
                ops.lora_delta(out, x, a_stack, b_stack, CTX.token_slots, scales, spans)
            return out
        for proj in projs:
            stacks = _get_stacks(layer_idx, [proj], x.shape[1], x.dtype, x.device)
            if stacks is None:
                continue
            a_stack, b_stack, scales, _ = stacks
            ops.lora_bgmv(out, x, a_stack, b_stack, CTX.token_slots, scales, proj[1])
        return out
    token_ids = CTX.token_lora_ids
    for lora_id, adapter in CTX.adapters.items():
        sel = (token_ids == lora_id).nonzero(as_tuple=True)[0]
        if sel.numel() == 0:
            continue
        x_sub = x[sel]
        for name, start, end in projs:
            ab = adapter.weights.get((layer_idx, name))
            if ab is None:
                continue
            a, b = ab
            delta = (x_sub @ a.t()) @ b.t()
            out[sel, start:end] += (delta * adapter.scaling).to(out.dtype)
    return out


def load_lora_adapter(
    path: str,
    lora_int_id: int,
    *,
    device: str,
    dtype: torch.dtype,
    max_lora_rank: int,
) -> LoRAAdapter:
    cfg_path = os.path.join(path, "adapter_config.json")
    with open(cfg_path) as f:
        cfg = json.load(f)
    if cfg.get("peft_type") != "LORA":
        raise ValueError(f"unsupported peft_type {cfg.get('peft_type')}")
    r = int(cfg["r"])
    if r > max_lora_rank:
        raise ValueError(f"LoRA rank {r} exceeds max_lora_rank {max_lora_rank}")
    alpha = float(cfg.get("lora_alpha", r))
    scaling = alpha / r

    weights_file = os.path.join(path, "adapter_model.safetensors")
    if os.path.exists(weights_file):
        from safetensors.torch import load_file

        raw = load_file(weights_file)
    else:
        bin_file = os.path.join(path, "adapter_model.bin")
        raw = torch.load(bin_file, map_location="cpu", weights_only=True)

    tp = get_tp_world_size()
    rank_idx = get_tp_rank()
    weights: dict[tuple[int, str], tuple[torch.Tensor, torch.Tensor]] = {}
    pending: dict[tuple[int, str], dict[str, torch.Tensor]] = {}
    for key, tensor in raw.items():
        # e.g. base_model.model.model.layers.3.self_attn.q_proj.lora_A.weight
        parts = key.split(".")
        try:
            li = parts.index("layers")
            layer_idx = int(parts[li + 1])
        except (ValueError, IndexError):
            continue
        proj = next((p for p in parts if p in _SUPPORTED), None)
        if proj is None:
            continue
        ab = "A" if "lora_A" in key else ("B" if "lora_B" in key else None)
        if ab is None:
            continue
        pending.setdefault((layer_idx, proj), {})[ab] = tensor

    for (layer_idx, proj), d in pending.items():
        if "A" not in d or "B" not in d:
            continue
        a = d["A"].to(torch.float32)  # [r, in]
        b = d["B"].to(torch.float32)  # [out, r]
        if tp > 1:
            if proj in _COLUMN:
                shard = b.shape[0] // tp
                b = b[rank_idx * shard:(rank_idx + 1) * shard]
            else:
                shard = a.shape[1] // tp
                a = a[:, rank_idx * shard:(rank_idx + 1) * shard]
        weights[(layer_idx, proj)] = (
            a.to(device=device, dtype=dtype),
            b.to(device=device, dtype=dtype),
        )
    if not weights:
        raise ValueError(f"adapter at {path} has no supported LoRA weights")
    return LoRAAdapter(lora_int_id=lora_int_id, rank=r, scaling=scaling, weights=weights)
