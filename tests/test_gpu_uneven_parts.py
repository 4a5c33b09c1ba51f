"""The two launches over 64-token tiles with K parts that do not divide K (csrc/sgmv.hip), against fp64: parts of a single 64-column piece and
pieces that are not shared out evenly, every number of rank groups and of 16-token blocks, short segments, adapters below the buffers'
rank with NaN beyond it, buffers of a rank between the kernels' own, fp16 and bf16."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
LENGTHS = [1, 7, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 130]

# rank, K, parts, widths, element type, adapters of lower rank
CASES = [
    (8, 128, 2, [8], B16, False), (8, 1152, 4, [72, 1032], F16, True), (16, 384, 4, [264], F16, False), (16, 2560, 3, [512], B16, True), (24, 640, 3, [64, 200], B16, True),
    (32, 1920, 4, [136], B16, False), (32, 896, 3, [520, 64, 8], F16, True), (40, 2560, 3, [72], F16, False), (48, 1920, 4, [1288], B16, True), (56, 1152, 4, [64], F16, True),
    (64, 2560, 3, [1024], B16, False), (64, 640, 4, [256, 256, 72], F16, True), (64, 3200, 3, [72], B16, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_fp64(monkeypatch, case):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    rank, k, parts, widths, dtype, mixed = CASES[case]
    print(f"uneven parts {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    lengths = LENGTHS * 2 if mixed else LENGTHS
    slots = len(lengths)
    ids = [i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 9
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    below = [r for r in (1, 8, 9, 13, 16, 17, 24, 32, 33, 40, 47, 63) if r < rank]
    ranks = [pick.choice(below) if mixed and i % 4 else rank for i in range(slots)]
    shown_a, shown_b = [t.clone() for t in a], [t.clone() for t in b]  # what the oracle sees: zeros beyond a slot's rank
    for s, r in enumerate(ranks):
        for t, z in zip(a, shown_a):
            t[s, r:], z[s, r:] = float("nan"), 0
        for t, z in zip(b, shown_b):
            t[s, :, r:], z[s, :, r:] = float("nan"), 0
    dev = [t.cuda() for t in a], [t.cuda() for t in b]
    eff = torch.tensor(ranks, dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices.cuda(), slots)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    scratch = torch.full((_hip.add_workspace_bytes(tokens, len(widths), rank, dtype),), 255, dtype=torch.uint8, device="cuda")  # (sums start as NaN)
    _hip.workspace_init(scratch)
    part = 4 * tokens * len(widths) * rank
    written = []
    for name, value in (("MLORA_FORCE_FORM", _hip.FORM_SGMV), ("MLORA_SLAB", 0), ("MLORA_SGMV_KSPLIT", parts)):
        monkeypatch.setenv(name, str(value))
    _hip.reload_knobs()
    try:
        runs = []
        for _ in range(2):
            out = y.cuda()
            _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, _hip.FORM_AUTO, scratch, effective_rank=eff)
            runs.append(out.cpu())
        sums = scratch[-4 * part:].view(torch.float32).view(4, -1)  # (the workspace ends with room for four parts)
        written = [bool((~torch.isnan(s)).any()) for s in sums.cpu()]
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert written == [p < parts for p in range(4)]
    assert torch.equal(runs[0], runs[1])
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"uneven parts {CASES[case]}")
