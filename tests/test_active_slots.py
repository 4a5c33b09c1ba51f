"""What the library is told about how many slots have tokens (mlora_add_lora_active, on which AUTO's choice depends): the
number where the host counted it, 0 behind capacities and under capture, and the same results whatever it is."""

import types

import pytest
import torch

from nanovllm_voxcpm_amd.lora import HipLoRABackend, LoRAMetadata
from nanovllm_voxcpm_amd.lora_ops.segment_meta import known_active_slots, mark_capacity


def _metadata(context) -> LoRAMetadata:
    return LoRAMetadata(context.token_to_slot, context.token_indices_sorted_by_slot, context.active_slot_ids, context.num_tokens_per_slot,
                        context.slot_start_offsets, context.no_lora_flag, context.num_active_loras)


def test_capacities_and_captured_counts_are_not_known_counts():
    ids = torch.arange(3, dtype=torch.int32)
    meta = LoRAMetadata(None, None, ids, None, None, False, 3)
    assert known_active_slots(meta, 8, 0) == 3 and known_active_slots(meta, 8, None) == 3
    assert known_active_slots(meta, 8, 5) == 0  # captured
    assert known_active_slots(meta, 2, 0) == 0  # more than there are slots
    assert known_active_slots(types.SimpleNamespace(), 8, 0) == 0
    mark_capacity(ids)
    assert known_active_slots(meta, 8, 0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("python_path", [False, True])
def test_the_library_is_told_what_the_host_counted(monkeypatch, python_path):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.engine.graph_meta import make_graph_domain_buffers, set_graph_lora_contexts
    from nanovllm_voxcpm_amd.engine.lora_manager import build_lora_context_from_slot_list
    from nanovllm_voxcpm_amd.utils.context import LM_LORA_DOMAIN, LORA_DOMAINS, LoRAContext, build_lora_context_from_token_to_slot, get_lora_context

    slots, rank, k, n, ids = 8, 16, 256, 64, [5, 5, -1, 2, 5]
    a, b = torch.zeros(slots, rank, k, device="cuda", dtype=torch.bfloat16), torch.zeros(slots, n, rank, device="cuda", dtype=torch.bfloat16)
    x, y = torch.zeros(len(ids), k, device="cuda", dtype=torch.bfloat16), torch.zeros(len(ids), n, device="cuda", dtype=torch.bfloat16)
    backend, told = HipLoRABackend(), []
    if python_path:
        backend._fastcall = None
    else:  # (what the later calls of the step pass on)
        module = backend._fastcall
        backend._fastcall = types.SimpleNamespace(**{f: getattr(module, f) for f in dir(module) if not f.startswith("__")})
        backend._fastcall.set_step = lambda *args: (told.append(args[-1]), module.set_step(*args))
    launch = _hip.call_add_lora
    monkeypatch.setattr(_hip, "call_add_lora", lambda args, active: (told.append(active), launch(args, active)))

    def call(context):
        told.clear()
        meta = _metadata(context)
        backend.add_lora([y], x, [a], [b], indices=meta.token_to_slot, metadata=meta, scaling=1.0)
        return set(told)

    vector = torch.tensor(ids, dtype=torch.int32, device="cuda")
    exact = build_lora_context_from_slot_list(ids, max_slots=slots, device="cuda:0")
    assert call(exact) == {2}
    assert call(build_lora_context_from_token_to_slot(vector, max_slots=slots)) == {2}
    assert call(build_lora_context_from_token_to_slot(vector, max_slots=slots, sync=False)) == {0}
    buffers = {"lora_domains": {d: make_graph_domain_buffers(len(ids), slots + 1, "cuda") for d in LORA_DOMAINS}}
    contexts = {d: LoRAContext() for d in LORA_DOMAINS}
    contexts[LM_LORA_DOMAIN] = exact
    set_graph_lora_contexts(buffers, contexts)
    assert call(get_lora_context(LM_LORA_DOMAIN)) == {0}
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        assert call(exact) == {0}


# tokens, slots, slots in use, rank, K, widths: on both sides of each line that AUTO draws by the count
@pytest.mark.gpu
@pytest.mark.parametrize("tokens,slots,used,rank,k,widths", [
    (37, 8, 1, 32, 1024, [1024]),
    (37, 8, 4, 32, 1024, [512, 512]),
    (37, 8, 5, 32, 1024, [512, 512]),
    (64, 4, 4, 16, 1024, [1024]),
    (65, 4, 4, 16, 1024, [1024]),
    (40, 32, 16, 64, 4096, [1024]),
    (40, 31, 15, 64, 4096, [1024]),
])
def test_a_known_count_changes_the_form_and_not_the_result(tokens, slots, used, rank, k, widths):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan
    from test_gpu_parity import _check, _exact

    print(f"{tokens} tokens, {used} of {slots} slots, rank {rank}, K {k}", flush=True)
    g = torch.Generator().manual_seed(tokens + slots)
    indices = ((torch.arange(tokens, dtype=torch.int32) * used // tokens) * (slots // used)).cuda()
    assert indices.unique().numel() == used
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).bfloat16().cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).bfloat16().cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).bfloat16().cuda(), torch.randn(tokens, sum(widths), generator=g).bfloat16().cuda()
    cols = [sum(widths[:i]) for i in range(len(widths))]
    exact, mag = _exact(types.SimpleNamespace(a=a, b=b, widths=widths), x, y, indices)
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, torch.bfloat16) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    for active in (0, used):
        out = y.clone()
        _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 1.0, _hip.FORM_AUTO, scratch, active_slots=active)
        _check(out, y, exact, mag, indices, f"{active} slots known")
