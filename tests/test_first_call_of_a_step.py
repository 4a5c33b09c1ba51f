"""The first call of a step in C++: taken where the step's slot vector carries the plan of the launch that made it and nothing
else is new, with the bits of the Python path; left to Python for everything else."""

import pytest
import torch

from nanovllm_voxcpm_amd.lora import HipLoRABackend, LoRAMetadata

SLOTS, RANK, K, N = 6, 16, 256, 64


def _metadata(context, slots=None):
    return LoRAMetadata(
        token_to_slot=context.token_to_slot if slots is None else slots,
        token_indices_sorted_by_slot=context.token_indices_sorted_by_slot,
        active_slot_ids=context.active_slot_ids,
        num_tokens_per_slot=context.num_tokens_per_slot,
        slot_start_offsets=context.slot_start_offsets,
        no_lora_flag=False,
        num_active_loras=context.num_active_loras,
    )


class _Calls:
    """One layer's buffers under two backends, the second without the C++ host path."""

    def __init__(self):
        g = torch.Generator().manual_seed(5)
        self.a = (torch.randn(SLOTS, RANK, K, generator=g) * 0.05).bfloat16().cuda()
        self.b = (torch.randn(SLOTS, N, RANK, generator=g) * 0.1).bfloat16().cuda()
        self.x, self.y = torch.randn(40, K, generator=g).bfloat16().cuda(), torch.randn(40, N, generator=g).bfloat16().cuda()
        self.backend, self.python = HipLoRABackend(), HipLoRABackend()
        self.python._fastcall = None

    def counters(self):
        return self.backend._fastcall.counters(self.backend._fast_state())

    def run(self, meta, rows):
        outs = []
        for backend in (self.python, self.backend):
            y = self.y[:rows].clone()
            backend.add_lora([y], self.x[:rows], [self.a], [self.b], indices=meta.token_to_slot, metadata=meta, scaling=1.0)
            outs.append(y.cpu())
        assert torch.equal(*outs)
        return outs[1]


def _context(ids):
    from nanovllm_voxcpm_amd.engine.lora_manager import build_lora_context_from_slot_list

    return build_lora_context_from_slot_list(ids, max_slots=SLOTS, device="cuda:0")


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 33])
def test_taken_with_the_plan_that_came_along(rows):
    calls = _Calls()
    calls.run(_metadata(_context([1] * 40)), 40)  # the buffers become known
    handled, passed = calls.counters()
    results = []
    for step in range(1, 5):
        ids = [((i + 1) * step) % (SLOTS + 1) - 1 for i in range(rows)]
        meta = _metadata(_context(ids))  # (all of the step's objects may be gone before its kernels have run)
        results.append(calls.run(meta, rows))
        assert calls.counters() == (handled + step, passed)
    assert rows == 1 or not torch.equal(results[0], results[1])


@pytest.mark.gpu
def test_left_to_python_when_anything_differs():
    from nanovllm_voxcpm_amd.utils.context import invalidate_lora_context

    calls = _Calls()
    first = calls.run(_metadata(_context([1] * 40)), 40)
    handled, passed = calls.counters()

    def passes_on(meta, rows):
        before = calls.counters()
        out = calls.run(meta, rows)
        assert calls.counters() == (before[0], before[1] + 1)
        return out

    passes_on(_metadata(_context([1] * 40)), 39)  # fewer rows than the vector has
    context = _context([0] * 40)
    rewritten = context.token_to_slot
    rewritten.fill_(1)  # the version moves on: the plan that came along is of other ids
    assert torch.equal(passes_on(_metadata(context), 40), first)
    context = _context([0] * 40)
    context.token_to_slot.data.fill_(1)  # (a write that nobody counts, announced by hand)
    invalidate_lora_context(context)
    assert torch.equal(passes_on(_metadata(context), 40), first)
    context = _context([1] * 40)
    assert torch.equal(passes_on(_metadata(context, context.token_to_slot.clone()), 40), first)  # no plan came with the copy
    # a context made for another number of slots than the buffers have
    from nanovllm_voxcpm_amd.engine.lora_manager import build_lora_context_from_slot_list
    passes_on(_metadata(build_lora_context_from_slot_list([1] * 40, max_slots=SLOTS + 2, device="cuda:0")), 40)
    # another stream: its scratch buffer is not known
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        assert torch.equal(passes_on(_metadata(_context([1] * 40)), 40), first)
    stream.synchronize()
    # a step that was taken here and is then captured: the plan is built inside the graph
    context = _context([1] * 40)
    meta = _metadata(context)
    assert torch.equal(calls.run(meta, 40), first)
    y, graph = calls.y.clone(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    before = calls.counters()
    with torch.cuda.graph(graph):
        calls.backend.add_lora([y], calls.x, [calls.a], [calls.b], indices=meta.token_to_slot, metadata=meta, scaling=1.0)
    assert calls.counters() == (before[0], before[1] + 1)
    for slot in (1, 4):
        meta.token_to_slot.fill_(slot)
        y.copy_(calls.y)
        graph.replay()
        assert torch.equal(y.cpu(), calls.run(_metadata(_context([slot] * 40)), 40))
