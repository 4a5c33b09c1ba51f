"""The segment plan that a batch context's slot vector brings along (segment_meta.attach_plan) serves the vector it was
built from and no rewritten one: rewrites that the version counter sees, and rewrites that it does not see and that
are announced by invalidating or installing the context."""

import copy
import dataclasses

import pytest
import torch

from nanovllm_voxcpm_amd.lora import HipLoRABackend, LoRAMetadata
from nanovllm_voxcpm_amd.lora_ops import segment_meta
from nanovllm_voxcpm_amd.utils.context import LoRAContext, invalidate_lora_context, set_lora_context

SLOTS = 4


def _metadata(context: LoRAContext) -> LoRAMetadata:
    return LoRAMetadata(context.token_to_slot, None, None, None, None, False, 1)


@pytest.fixture
def built(monkeypatch):
    """Plans built so far; nothing here needs a GPU."""
    calls = []

    def build(tts, max_slots):
        calls.append(tts)
        return segment_meta.SegmentPlan(torch.full((16,), len(calls), dtype=torch.int32), tts, tts.numel(), max_slots)

    monkeypatch.setattr("nanovllm_voxcpm_amd.lora.build_segment_plan", build)
    monkeypatch.setattr(segment_meta._hip, "stream_capture_id", lambda *_: 0)
    return calls


def _attached() -> tuple[LoRAContext, torch.Tensor]:
    tts = torch.tensor([0, 1, 2, 3, 0], dtype=torch.int32)
    workspace = torch.zeros(16, dtype=torch.int32)
    segment_meta.attach_plan(tts, workspace, SLOTS)
    return LoRAContext(token_to_slot=tts, no_lora_flag=False, num_active_loras=4), workspace


def test_attached_plan_serves_the_vector_it_was_built_from(built):
    context, workspace = _attached()
    tts = context.token_to_slot
    assert HipLoRABackend._plan_for(_metadata(context), tts, SLOTS, 0).workspace is workspace and not built
    # another number of slots, part of the vector, a capture in progress
    assert HipLoRABackend._plan_for(_metadata(context), tts, SLOTS + 1, 0).workspace is not workspace
    assert HipLoRABackend._plan_for(_metadata(context), tts[:3], SLOTS, 0).workspace is not workspace
    assert HipLoRABackend._plan_for(_metadata(context), tts, SLOTS, 7).workspace is not workspace
    assert len(built) == 3


@pytest.mark.parametrize("announce", [invalidate_lora_context, set_lora_context, None])
def test_attached_plan_goes_with_a_rewrite(built, announce):
    context, workspace = _attached()
    tts = context.token_to_slot
    if announce is None:
        tts.copy_(tts.flip(0))
    else:
        version = tts._version
        tts.data.copy_(tts.flip(0))  # (the counter does not see this one)
        assert tts._version == version
        announce(context)
    assert HipLoRABackend._plan_for(_metadata(context), tts, SLOTS, 0).workspace is not workspace
    assert len(built) == 1


def _built(workspace: torch.Tensor) -> LoRAContext:
    from nanovllm_voxcpm_amd.engine.lora_manager import _with_plan

    return _with_plan(torch.tensor([0, 1, 2, 3, 0], dtype=torch.int32), workspace, SLOTS, no_lora_flag=False, num_active_loras=4)


@pytest.mark.parametrize("first", [None, lambda c: c.token_to_slot, copy.copy, copy.deepcopy, dataclasses.replace, repr, invalidate_lora_context,
                                   set_lora_context])
def test_the_plan_survives_an_installation_only_while_nobody_could_have_rewritten_the_vector(built, first):
    workspace = torch.zeros(16, dtype=torch.int32)
    context = _built(workspace)
    if first is not None:
        first(context)
    set_lora_context(context)
    plan = HipLoRABackend._plan_for(_metadata(context), context._slots, SLOTS, 0)
    assert (plan.workspace is workspace) == (first is None) and len(built) == (first is not None)


@pytest.mark.gpu
@pytest.mark.parametrize("announce", [invalidate_lora_context, set_lora_context])
def test_tokens_follow_a_slot_vector_rewritten_past_its_version_counter(announce):
    from nanovllm_voxcpm_amd.engine.lora_manager import build_lora_context_from_slot_list
    from oracle import lora_apply as oracle

    tokens, k, n, rank = 70, 256, 64, 16
    g = torch.Generator().manual_seed(5)
    ids = [(3 * i) % (SLOTS + 1) - 1 for i in range(tokens)]
    x, y = torch.randn(tokens, k, generator=g).bfloat16(), torch.randn(tokens, n, generator=g).bfloat16()
    a, b = (torch.randn(SLOTS, rank, k, generator=g) * 0.05).bfloat16(), (torch.randn(SLOTS, n, rank, generator=g) * 0.1).bfloat16()
    torch.zeros(1, device="cuda")
    context = build_lora_context_from_slot_list(ids, max_slots=SLOTS, device="cuda:0")
    backend, dev = HipLoRABackend(), [t.cuda() for t in (x, a, b)]
    for now in (ids, ids[::-1]):
        if now is not ids:
            context.token_to_slot.data.copy_(torch.tensor(now, dtype=torch.int32))
            announce(context)
        out = y.cuda()
        backend.add_lora([out], dev[0], [dev[1]], [dev[2]], indices=context.token_to_slot, metadata=_metadata(context), scaling=1.0)
        slots = torch.tensor(now, dtype=torch.int32)
        (want,) = oracle.fused_add_lora([y], x, [a], [b], indices=slots, scaling=1.0, accumulate=torch.float64)
        assert torch.equal(out.cpu()[slots < 0], y[slots < 0])
        assert torch.allclose(out.cpu().float(), want.float(), rtol=2**-7, atol=2**-8)
