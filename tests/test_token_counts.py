"""What the library is told about how many tokens have a slot (mlora_add_lora_counts): as many as the context lists where its counts are the
batch's own, else 0; how a launch is cut changes with it (ranges of 512, 1024 or 2048 columns, parts of K), its results do not."""

import types

import pytest
import torch

from nanovllm_voxcpm_amd.lora import LoRAMetadata
from nanovllm_voxcpm_amd.lora_ops.segment_meta import known_active_tokens, mark_capacity


def test_only_the_batch_s_own_list_is_a_known_count():
    ids, listed = torch.arange(3, dtype=torch.int32), torch.arange(7)
    meta = LoRAMetadata(None, listed, ids, None, None, False, 3)
    assert known_active_tokens(meta, 8, 9, 0) == 7 and known_active_tokens(meta, 8, 7, None) == 7
    assert known_active_tokens(meta, 8, 6, 0) == 0  # more than there are rows
    assert known_active_tokens(meta, 8, 9, 5) == 0  # captured
    assert known_active_tokens(meta, 2, 9, 0) == 0  # more slots than there are
    assert known_active_tokens(types.SimpleNamespace(), 8, 9, 0) == 0
    assert known_active_tokens(types.SimpleNamespace(num_active_loras=3, token_indices_sorted_by_slot=[1, 2]), 8, 9, 0) == 0
    mark_capacity(ids)
    assert known_active_tokens(meta, 8, 9, 0) == 0


# rank, K, widths, tokens, slots: ranges of 512 or 1024 columns, of up to 2048, and of a batch of short segments
@pytest.mark.gpu
@pytest.mark.parametrize("rank,k,widths,tokens,slots", [
    (64, 256, [1032, 520], 5200, 2),
    (16, 2048, [2056], 4700, 3),
    (32, 128, [4104], 2100, 33),
])
def test_a_known_count_changes_the_cut_and_not_the_result(rank, k, widths, tokens, slots):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan
    from test_gpu_parity import _check, _exact

    print(f"rank {rank}, K {k}, {widths}, {tokens} tokens of {slots} slots", flush=True)
    g = torch.Generator().manual_seed(tokens)
    indices = (torch.arange(tokens, dtype=torch.int32) * slots // tokens)
    indices[::5] = -1
    used = int((indices >= 0).sum())
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).bfloat16().cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).bfloat16().cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).bfloat16().cuda(), torch.randn(tokens, sum(widths), generator=g).bfloat16().cuda()
    cols = [sum(widths[:i]) for i in range(len(widths))]
    indices = indices.cuda()
    exact, mag = _exact(types.SimpleNamespace(a=a, b=b, widths=widths), x, y, indices)
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, torch.bfloat16) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    for form in (_hip.FORM_WIDE, _hip.FORM_SGMV, _hip.FORM_AUTO):
        for count in (0, used, 1, 64 * slots, tokens + 5):  # (a wrong one costs time and nothing else)
            out = y.clone()
            _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 1.0, form, scratch, active_slots=slots if count else 0, active_tokens=count)
            _check(out, y, exact, mag, indices, f"form {form}, {count} tokens known")
