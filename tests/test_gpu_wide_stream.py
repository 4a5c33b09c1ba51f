"""One launch over 64-token tiles as one stream of stages (csrc/wide.hip) against fp64 at the sizes where it can go wrong: every rank of the buffers with
adapters in every group of ranks (NaN beyond them), tiles of every number of 16-token blocks and barely started ones, short segments, K of
fewer chunks than a stage holds and chunks that do not fill the last stage, ranges of fewer spans than a stage holds and spans that end early."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
LENGTHS = [1, 7, 15, 16, 17, 31, 32, 33, 48, 49, 63, 64, 65, 130]

# rank, K, widths, element type, adapters of lower rank
CASES = [
    (8, 128, [8], B16, False), (8, 640, [72, 1032], F16, True), (16, 128, [512], F16, False), (16, 384, [64, 200], B16, True),
    (32, 128, [136], B16, False), (32, 640, [520, 64], F16, True), (64, 128, [8], F16, False), (64, 256, [1024, 256, 256], B16, True),
    (64, 1152, [576], B16, True), (64, 4096, [72], F16, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_fp64(case):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    rank, k, widths, dtype, mixed = CASES[case]
    print(f"wide stream {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    lengths = LENGTHS * 2 if mixed else LENGTHS
    slots = len(lengths)
    ids = [i for i, n in enumerate(lengths) for _ in range(n)] + [-1] * 9
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    below = [r for r in (1, 8, 9, 13, 16, 17, 24, 32, 33, 40, 63) if r < rank]
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
    runs = []
    for _ in range(2):
        out = y.cuda()
        _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, _hip.FORM_WIDE, effective_rank=eff)
        runs.append(out.cpu())
    assert torch.equal(runs[0], runs[1])
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"wide stream {CASES[case]}")
