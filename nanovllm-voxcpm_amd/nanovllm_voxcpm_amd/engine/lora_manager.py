"""Batch plan -> device LoRA context, with the segment arrays built on the GPU.

Counterpart of the index builders of the reference's ``nanovllm_voxcpm/engine/lora_manager.py``
(:67-180).  The reference sorts the tokens by slot in Python for every step and domain
(:77-91) and uploads five packed arrays (:118-176); here the slot ids travel with the launch of the
on-device counting sort (those of very many sequences through one pinned copy), which produces the rest.  The
adapter lifecycle / LRU residency half of that file lives in ``lora_runtime.py`` and is
re-exported here under the reference's import path.
"""

from __future__ import annotations

from array import array

import numpy as np
import torch

from nanovllm_voxcpm_amd import _hip
from nanovllm_voxcpm_amd.lora_ops.segment_meta import attach_plan
from nanovllm_voxcpm_amd.utils.context import LoRAContext


class LoRABatchPlan:
    """What the scheduler knows on the host: which slot every token of the batch uses.

    Takes the six fields of the reference's dataclass (lora_manager.py:67-75) in its order; the
    four segment arrays may be left out and are then derived from ``token_to_slot`` on demand
    (the device path never reads them: the GPU sorts the tokens itself)."""

    __slots__ = ("adapter_to_slot", "_tokens", "_runs", "_sorted", "_active", "_counts", "_offsets")

    def __init__(
        self,
        adapter_to_slot: dict[int, int],
        token_to_slot: list[int],
        token_indices_sorted_by_slot: list[int] | None = None,
        active_slot_ids: list[int] | None = None,
        num_tokens_per_slot: list[int] | None = None,
        slot_start_offsets: list[int] | None = None,
    ) -> None:
        self.adapter_to_slot = adapter_to_slot
        self._tokens: list[int] | None = token_to_slot
        self._runs: tuple[list[int], list[int]] | None = None
        self._sorted = token_indices_sorted_by_slot
        self._active = active_slot_ids
        self._counts = num_tokens_per_slot
        self._offsets = slot_start_offsets

    @classmethod
    def from_runs(cls, adapter_to_slot: dict[int, int], slots: list[int], counts: list[int]) -> "LoRABatchPlan":
        """The plan of a batch known per sequence (slot id and token count): the per-token list, which
        the device path does not need, is only written out when somebody asks for it."""
        plan = cls(adapter_to_slot, None)  # type: ignore[arg-type]
        plan._runs = (slots, counts)
        return plan

    @property
    def token_to_slot(self) -> list[int]:
        if self._tokens is None:  # from here on the list, which the caller may edit, is what counts
            self._tokens, self._runs = expand_token_to_slot(*self._runs), None
        return self._tokens

    @token_to_slot.setter
    def token_to_slot(self, tokens: list[int]) -> None:
        self._tokens, self._runs = tokens, None

    def _listed(self) -> list[int]:
        """The per-token slot ids for reading: not handed out, so the runs stay in force."""
        return self._tokens if self._tokens is not None else expand_token_to_slot(*self._runs)

    def runs(self) -> tuple[list[int], list[int]]:
        """(slot ids, token counts) whose expansion is ``token_to_slot``."""
        return self._runs if self._runs is not None else (self._tokens, [1] * len(self._tokens))

    def __repr__(self) -> str:
        return f"LoRABatchPlan(adapter_to_slot={self.adapter_to_slot!r}, token_to_slot={self._listed()!r})"

    def __eq__(self, other) -> bool:
        if not isinstance(other, LoRABatchPlan):
            return NotImplemented
        return self.adapter_to_slot == other.adapter_to_slot and list(self._listed()) == list(other._listed())

    @property
    def num_lora_tokens(self) -> int:
        slots, counts = self.runs()
        without = sum([c for s, c in zip(slots, counts) if s < 0]) if min(slots, default=0) < 0 else 0
        return sum(counts) - without

    @property
    def active_slot_ids(self) -> list[int]:
        if self._active is None:
            self._active = self._used_slots()
        return self._active

    def _used_slots(self) -> list[int]:
        slots, counts = self.runs()
        used = set(slots) if 0 not in counts else {s for s, c in zip(slots, counts) if c > 0}
        return sorted([s for s in used if s >= 0])

    @property
    def num_tokens_per_slot(self) -> list[int]:
        if self._counts is None:
            tokens = self._listed()
            self._counts = [sum(1 for s in tokens if s == slot) for slot in self.active_slot_ids]
        return self._counts

    @property
    def slot_start_offsets(self) -> list[int]:
        if self._offsets is None:
            offsets = [0]
            for count in self.num_tokens_per_slot:
                offsets.append(offsets[-1] + count)
            self._offsets = offsets
        return self._offsets

    @property
    def token_indices_sorted_by_slot(self) -> list[int]:
        if self._sorted is None:
            keyed = [(s, t) for t, s in enumerate(self._listed()) if s >= 0]
            self._sorted = [t for _, t in sorted(keyed)]
        return self._sorted


def build_lora_batch_plan_from_token_to_slot(
    adapter_to_slot: dict[int, int],
    token_to_slot: list[int],
) -> LoRABatchPlan:
    return LoRABatchPlan(adapter_to_slot=adapter_to_slot, token_to_slot=list(token_to_slot))


def expand_token_to_slot(adapter_slots: list[int], token_counts: list[int]) -> list[int]:
    """Per-sequence slot ids repeated per token (reference: lora_manager.py:399-403)."""
    if len(adapter_slots) != len(token_counts):
        raise ValueError("adapter_ids and token_counts must have the same length")
    out: list[int] = []
    for slot, count in zip(adapter_slots, token_counts):
        out.extend([slot] * count)
    return out


def _pinned_slots(slots: list[int], counts: list[int], n: int) -> torch.Tensor:
    """The per-token slot ids expanded into a pinned buffer."""
    host = torch.empty(n, dtype=torch.int32, device="cpu", pin_memory=True)
    ids = np.frombuffer(array("i", slots), dtype=np.int32)
    host.numpy()[:] = ids if counts.count(1) == len(counts) else np.repeat(ids, np.frombuffer(array("q", counts), dtype=np.int64))
    return host


def _with_plan(tts: torch.Tensor, workspace: torch.Tensor, max_slots: int, **fields) -> LoRAContext:
    """A context over arrays made here, its slot vector with the segment plan of the same launch."""
    attach_plan(tts, workspace, max_slots)
    context = LoRAContext(token_to_slot=tts, **fields)
    context._unseen = True
    return context


def _context_in_one_launch(slots: list[int], counts: list[int], max_slots: int | None, device: torch.device | str) -> LoRAContext | None:
    """The context of a batch whose runs fit the arguments of the metadata launch; None (nothing done) for others."""
    fast = _hip.load_fastcall()
    if fast is None or not torch.cuda.is_initialized():
        return None
    totals = fast.run_totals(slots, counts)
    if totals is None:
        return None
    n, n_lora, n_active, largest = totals
    if max_slots is None:
        max_slots = largest + 1
    if n_active == 0 or largest >= max_slots:
        return None
    cap = min(n, max_slots)
    # slot vector | sorted indices | ids | counts | offsets | plan (its start on a 256-byte boundary)
    head = (2 * n + 3 * cap + 1 + 63) & ~63
    words = _hip.plan_workspace_words(n, max_slots)
    packed = torch.empty(head + words, dtype=torch.int32, device=device)
    index = packed.device.index
    if index is None or index != _hip.current_device_index():
        return None
    tts, sorted_idx, _, ids, _, per_slot, _, offsets, _, workspace = packed.split_with_sizes(
        [n, n_lora, n - n_lora, n_active, cap - n_active, n_active, cap - n_active, n_active + 1, head - 2 * n - 2 * cap - n_active - 1, words])
    at = packed.data_ptr()
    rc = fast.build_context(_hip.entry_point("mlora_meta_build_runs"), slots, counts, index, max_slots, cap, at, at + 4 * n, at + 8 * n,
                            at + 8 * n + 4 * cap, at + 8 * n + 8 * cap, at + 4 * head)
    _hip._check(rc, "mlora_meta_build_runs")
    return _with_plan(tts, workspace, max_slots, token_indices_sorted_by_slot=sorted_idx, active_slot_ids=ids, num_tokens_per_slot=per_slot,
                      slot_start_offsets=offsets, no_lora_flag=False, num_active_loras=n_active)


def build_lora_context_from_batch_plan(
    plan: LoRABatchPlan,
    *,
    max_slots: int | None = None,
    device: torch.device | str = "cuda",
) -> LoRAContext:
    """One metadata launch, no device->host traffic: the array lengths and the two host flags come
    from the host list the plan already holds.  A second workgroup of the launch builds the segment
    plan of eager calls, which costs no time of its own.  The slot ids travel with the launch, those of batches
    of very many sequences through one H2D copy ahead of it."""
    slots, counts = plan.runs()
    context = _context_in_one_launch(slots, counts, max_slots, device)
    if context is not None:
        return context
    n = sum(counts)
    active = plan._used_slots()
    if not active:
        tts = _pinned_slots(slots, counts, n).to(device, non_blocking=True) if n else torch.empty(0, dtype=torch.int32, device=device)
        return LoRAContext(token_to_slot=tts, no_lora_flag=True, num_active_loras=0)
    n_lora, n_active = plan.num_lora_tokens, len(active)
    if max_slots is None:
        max_slots = active[-1] + 1
    elif active[-1] >= max_slots:
        raise ValueError(f"slot id {active[-1]} is outside the {max_slots} resident slots")
    cap = min(n, max_slots)
    # one allocation: slot vector, index arrays, segment plan (its start on a 256-byte boundary)
    head = (2 * n + 2 * cap + cap + 1 + 63) & ~63
    packed = torch.empty(head + _hip.plan_workspace_words(n, max_slots), dtype=torch.int32, device=device)
    tts, sorted_idx, ids, per_slot, offsets = packed[: 2 * n + 2 * cap + cap + 1].split([n, n, cap, cap, cap + 1])
    tts.copy_(_pinned_slots(slots, counts, n), non_blocking=True)
    workspace = packed[head:]
    _hip.meta_build_many([
        dict(token_to_slot=tts, max_slots=max_slots, sorted_idx=sorted_idx, compact_ids=ids, compact_counts=per_slot,
             compact_offsets=offsets, compact_capacity=cap),
        dict(token_to_slot=tts, max_slots=max_slots, plan=workspace),
    ])
    return _with_plan(
        tts,
        workspace,
        max_slots,
        token_indices_sorted_by_slot=sorted_idx[:n_lora],
        active_slot_ids=ids[:n_active],
        num_tokens_per_slot=per_slot[:n_active],
        slot_start_offsets=offsets[: n_active + 1],
        no_lora_flag=False,
        num_active_loras=n_active,
    )


def build_lora_context_from_slot_list(
    token_to_slot: list[int],
    *,
    max_slots: int | None = None,
    device: torch.device | str = "cuda",
) -> LoRAContext:
    return build_lora_context_from_batch_plan(
        build_lora_batch_plan_from_token_to_slot({}, token_to_slot), max_slots=max_slots, device=device
    )


from nanovllm_voxcpm_amd.engine.lora_runtime import (  # noqa: E402  (re-export under the reference's module path)
    LoRAControlEntry,
    LoRALifecycleState,
    LoRAManager,
    LoRAModelPayload,
    LoRAModulePayload,
    LoRAResidentState,
    LoRARuntime,
    LoRARuntimeEntry,
    LoRASlot,
)
