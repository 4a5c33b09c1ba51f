"""Launches with the non-temporal hint leave the bits of those without.  The expand over 64-token tiles with it on y
(csrc/sgmv.hip): every rank, one tile and two per workgroup, tiles that end inside a 16-token block, column counts that end
inside a span, adapters below the buffers' rank, tokens without an adapter.  The pair over 16-token tiles with it on A and B
(csrc/pair.hip): slots of one tile beside slots of several, every number of row groups, both element sizes."""

import random

import pytest
import torch

B16, F16 = torch.bfloat16, torch.float16

# segment lengths, rank, K, widths, tiles per workgroup, element type, adapters of lower rank
CASES = [
    ([64], 8, 128, [8], 1, B16, False),
    ([130, 65, 1, 15], 16, 256, [520, 64], 2, F16, False),
    ([33, 200, 3], 32, 128, [1032], 2, B16, True),
    ([65, 63, 300, 17], 64, 256, [4096, 264], 2, B16, True),
    ([1, 500, 49], 64, 128, [2048], 1, F16, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_hint_changes_no_bit(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    lengths, rank, k, widths, group, dtype, mixed = CASES[case]
    print(f"stream hint {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    slots = len(lengths)
    ids = [i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 5
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32, device="cuda"), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype).cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype).cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype).cuda(), torch.randn(tokens, sum(widths), generator=g).to(dtype).cuda()
    eff = torch.tensor([pick.choice([1, 5, 8, rank // 2, rank]) for _ in range(slots)], dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, dtype), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    runs = []
    try:
        for hint in (0, 1):
            monkeypatch.setenv("MLORA_SGMV_STREAM", str(hint))
            monkeypatch.setenv("MLORA_SGMV_GROUP", str(group))
            _hip.reload_knobs()
            out = y.clone()
            _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 0.75, _hip.FORM_SGMV, scratch, effective_rank=eff)
            runs.append(out)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(*runs) and not torch.equal(runs[0], y)
    assert torch.equal(runs[0][indices < 0], y[indices < 0])


@pytest.mark.gpu
@pytest.mark.parametrize("rank, k, widths, dtype", [
    (8, 128, [8], B16), (16, 4096, [264], F16), (24, 1024, [520, 64], B16), (48, 2048, [256], F16), (64, 1024, [1024, 256, 256], B16),
    (16, 1024, [264], torch.float32), (40, 96, [12], torch.float32), (64, 2048, [200], torch.float32),
])
def test_hint_on_weights_changes_no_bit(rank, k, widths, dtype, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    lengths = [1, 15, 16, 17, 4, 40, 0, 9]
    print(f"hint on weights {rank} {k} {widths} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rank)
    slots = len(lengths)
    indices = torch.tensor([i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 3, dtype=torch.int32, device="cuda")
    tokens = indices.numel()
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype).cuda() for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype).cuda() for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype).cuda(), torch.randn(tokens, sum(widths), generator=g).to(dtype).cuda()
    plan = build_segment_plan(indices, slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, dtype) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    form = _hip.FORM_AUTO if dtype == torch.float32 else _hip.FORM_PAIR  # (by name fp32 has fewer ranks)
    runs = []
    try:
        monkeypatch.setenv("MLORA_SOLO", "0")
        for hint in (0, 1):
            monkeypatch.setenv("MLORA_PAIR_ONCE", str(hint))
            _hip.reload_knobs()
            out = y.clone()
            _hip.add_lora(out, x, a, b, cols, indices, plan.workspace, 0.75, form, scratch)
            runs.append(out)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(*runs) and not torch.equal(runs[0], y)
