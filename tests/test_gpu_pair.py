"""The shrink / expand pair over 16-token tiles (csrc/pair.hip) at the sizes where it can go wrong: one
token, full and barely started tiles, K of one 128-byte chunk and of many parts, column counts that end
inside a span, every rank's B row length, adapters below the buffers' rank with NaN beyond it, fp32."""

import random
import types

import pytest
import torch

from oracle import lora_apply as oracle
from test_gpu_parity import _check, _exact

B16, F16, F32 = torch.bfloat16, torch.float16, torch.float32

# tokens, slots, rank, K, widths, element type, adapters of lower rank, segments instead of single tokens
CASES = [
    (1, 1, 8, 64, [8], B16, False, False),
    (16, 1, 8, 4096, [1032], B16, True, True),
    (7, 3, 16, 256, [64], B16, False, False),
    (17, 2, 24, 704, [520], F16, False, True),
    (64, 8, 32, 1024, [200, 72], F16, True, False),
    (40, 4, 40, 2048, [512], B16, False, False),
    (90, 5, 48, 1536, [1000, 24], B16, True, True),
    (33, 4, 56, 2048, [256, 64], F16, True, False),
    (200, 48, 64, 2048, [2048, 512, 512], F16, True, False),
    (300, 3, 64, 8192, [1024], B16, False, True),
    (1, 2, 8, 32, [4], F32, False, False),
    (77, 3, 64, 544, [1024, 64], F32, True, True),
    (257, 16, 32, 96, [8, 16, 24], F32, False, True),
    (40, 2, 16, 4096, [1024], F32, True, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_pair_form_against_fp64(case):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    tokens, slots, rank, k, widths, dtype, mixed, segments = CASES[case]
    print(f"pair {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    ids = []
    while len(ids) < tokens:
        ids += [pick.randrange(-1, slots)] * (pick.randrange(1, 70) if segments else 1)
    ids[0] = slots - 1
    indices = torch.tensor(ids[:tokens], dtype=torch.int32)
    a = [torch.randn(slots, rank, k, generator=g) * 0.05 for _ in widths]
    b = [torch.randn(slots, n, rank, generator=g) * 0.1 for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    ranks = [pick.choice([1, 5, 8, 13, rank // 2, rank]) if mixed else rank for _ in range(slots)]
    a, b = [t.to(dtype) for t in a], [t.to(dtype) for t in b]
    shown_a, shown_b = [t.clone() for t in a], [t.clone() for t in b]  # what the oracle sees: zeros beyond a slot's rank
    for s, r in enumerate(ranks):
        for t, z in zip(a, shown_a):
            t[s, r:], z[s, r:] = float("nan"), 0
        for t, z in zip(b, shown_b):
            t[s, :, r:], z[s, :, r:] = float("nan"), 0
    want = torch.cat(oracle.fused_add_lora(list(y.split(widths, dim=-1)), x, shown_a, shown_b, indices=indices, scaling=0.75,
                                           accumulate=torch.float64), dim=-1)
    dev = [t.cuda() for t in a], [t.cuda() for t in b]
    eff = torch.tensor(ranks, dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices.cuda(), slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, dtype) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    runs = []
    for _ in range(2):
        out = y.cuda()
        _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, _hip.FORM_PAIR, scratch, effective_rank=eff)
        runs.append(out.cpu())
    assert torch.equal(runs[0], runs[1])
    assert torch.equal(runs[0][indices < 0], y[indices < 0])
    if dtype == F32:
        assert torch.allclose(runs[0], want, rtol=1e-5, atol=2e-5)
    else:  # to one rounding of the exact sum and of the intermediate
        exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
        _check(runs[0], y, exact, mag, indices, f"pair {CASES[case]}")
