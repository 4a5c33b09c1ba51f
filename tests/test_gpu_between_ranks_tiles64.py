"""Buffers of a rank between the kernels' own (24, 40, 48, 56) over 64-token tiles, in one launch (csrc/wide.hip) and in two (csrc/sgmv.hip), against
fp64: A and B rows that end inside a kernel's block of ranks, the last slot's at the end of their buffers, adapters of every lower group of ranks
(NaN beyond them), tiles of every number of 16-token blocks, short segments, ranges and K that do not fill their last stage, and K parts."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
LENGTHS = [1, 7, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 130]

# rank, K, widths, element type, adapters of lower rank
CASES = [
    (24, 128, [8], B16, False), (24, 640, [72, 1032], F16, True), (24, 4096, [512], B16, True), (40, 384, [64, 200], B16, False), (40, 1152, [576], F16, True),
    (48, 256, [1024, 256, 256], B16, True), (48, 2048, [1288], B16, False), (48, 128, [4096, 4096], F16, True), (56, 640, [520, 64], F16, False),
    (56, 4096, [72], B16, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("form", [3, 8])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_fp64(monkeypatch, case, form):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    rank, k, widths, dtype, mixed = CASES[case]
    print(f"rank {rank} over 64-token tiles {CASES[case]}, form {form}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    lengths = LENGTHS * 2 if mixed else LENGTHS
    slots = len(lengths)
    ids = [i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 9
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    below = [r for r in (1, 8, 9, 13, 16, 17, 24, 32, 33, 40, 47) if r < rank]
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
    monkeypatch.setenv("MLORA_FORCE_FORM", str(form))
    _hip.reload_knobs()
    try:
        runs = []
        for _ in range(2):
            out = y.cuda()
            _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, _hip.FORM_AUTO, scratch, effective_rank=eff)
            runs.append(out.cpu())
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(runs[0], runs[1])
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"rank {rank} over 64-token tiles {CASES[case]}, form {form}")
    with pytest.raises(RuntimeError):  # by name, as before
        _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, form, scratch, effective_rank=eff)
