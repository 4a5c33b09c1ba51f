"""Metadata of a batch whose slot ids travel with the launch (mlora_meta_build_runs) at the edges of its table -
one run, the most runs, one token per run up to the most and one more, empty runs, runs without adapter -
against the integer oracle, the plan against the one built from the uploaded vector."""

import pytest
import torch

from oracle import segment_meta as oracle

CASES = {  # name: (slots, [(slot, count), ...])
    "one": (1, [(0, 1)]),
    "one_long": (4, [(3, 9392)]),
    "singles": (32, [((7 * i) % 33 - 1, 1) for i in range(1024)]),
    "singles_over": (32, [((7 * i) % 33 - 1, 1) for i in range(1025)]),
    "runs": (128, [((5 * i) % 129 - 1, i % 9) for i in range(336)]),
    "runs_over": (128, [((5 * i) % 129 - 1, i % 9) for i in range(337)]),
    "prompts": (16, [(2, 587), (-1, 63), (0, 0), (15, 1), (2, 700), (-1, 5)]),
    "none": (4, [(-1, 3), (1, 0)]),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_context_of_runs_bit_exact(name):
    from nanovllm_voxcpm_amd.engine.lora_manager import LoRABatchPlan, build_lora_context_from_batch_plan
    from nanovllm_voxcpm_amd.lora_ops import build_segment_plan

    max_slots, runs = CASES[name]
    print(f"runs {name}", flush=True)
    torch.zeros(1, device="cuda")  # (the runtime is up, as in a server)
    plan = LoRABatchPlan.from_runs({}, [s for s, _ in runs], [c for _, c in runs])
    context = build_lora_context_from_batch_plan(plan, max_slots=max_slots, device="cuda:0")
    tokens = [s for s, c in runs for _ in range(c)]
    assert plan.token_to_slot == tokens and context.token_to_slot.tolist() == tokens
    sorted_idx, ids, counts, offsets = oracle.engine_layout(tokens)
    assert context.no_lora_flag == (not ids)
    if not ids:
        return
    assert context.num_active_loras == len(ids)
    assert context.token_indices_sorted_by_slot.tolist() == list(sorted_idx) and context.active_slot_ids.tolist() == list(ids)
    assert context.num_tokens_per_slot.tolist() == list(counts) and context.slot_start_offsets.tolist() == list(offsets)
    workspace, slots, version = context.token_to_slot._mlora_plan
    assert (slots, version) == (max_slots, context.token_to_slot._version)
    want = build_segment_plan(context.token_to_slot.clone(), max_slots).workspace
    # (places that no list reaches hold whatever the allocation held: compared as the kernels read them)
    head = 16 + (len(tokens) + 3 & ~3)
    assert workspace[:16].tolist() == want[:16].tolist() and workspace[16 : 16 + len(sorted_idx)].tolist() == list(sorted_idx)
    assert workspace[head : head + max_slots + 1].tolist() == want[head : head + max_slots + 1].tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["singles", "singles_over", "runs", "runs_over"])
def test_a_context_and_its_plan_are_one_allocation(name):
    """What is recorded for the slot vector on another stream holds for everything the kernels read there."""
    from nanovllm_voxcpm_amd.engine.lora_manager import LoRABatchPlan, build_lora_context_from_batch_plan

    max_slots, runs = CASES[name]
    torch.zeros(1, device="cuda")
    context = build_lora_context_from_batch_plan(LoRABatchPlan.from_runs({}, [s for s, _ in runs], [c for _, c in runs]), max_slots=max_slots,
                                                 device="cuda:0")
    arrays = [context.token_to_slot, context.token_indices_sorted_by_slot, context.active_slot_ids, context.num_tokens_per_slot,
              context.slot_start_offsets, context.token_to_slot._mlora_plan[0]]
    assert len({t.untyped_storage().data_ptr() for t in arrays}) == 1
