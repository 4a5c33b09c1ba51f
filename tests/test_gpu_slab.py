"""The shrink over 64-token tiles through LDS (csrc/slab.hip) at the sizes where it can go wrong: tiles of every
number of 16-token blocks and barely started ones, short segments beside them, K parts of a single
128-byte piece per wavefront or less and uneven ones, every rank, adapters below the buffers' rank with NaN beyond it."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16

# segment lengths (slots in turn, every fourth without adapter when `holes`), rank, K, widths, K parts (0: the launch's
# own choice), element type, adapters of lower rank, holes
CASES = [
    ([64], 8, 128, [8], 0, B16, False, False),
    ([16, 17, 1, 15], 16, 128, [520, 64], 1, F16, False, False),
    ([32, 33, 48, 49, 3], 32, 384, [264], 3, B16, True, True),
    ([65, 63, 128, 7, 2, 300], 64, 1024, [1024, 256, 256], 0, B16, False, False),
    ([130, 20, 64, 31, 5], 64, 2048, [512], 4, F16, True, True),
    ([257, 16], 32, 4096, [1032], 2, B16, True, False),
    ([500, 40, 9], 16, 8192, [72, 200], 3, F16, False, True),
    ([300, 40], 32, 8192, [72], 0, B16, True, False),  # four parts from K = 8192 on
    ([4000, 4200], 16, 4096, [8], 0, F16, False, False),  # four parts of K = 4096 where tiles alone fill the chip
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_slab_shrink_against_fp64(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    lengths, rank, k, widths, parts, dtype, mixed, holes = CASES[case]
    print(f"slab {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    slots = len(lengths)
    ids = [-1 if holes and i % 4 == 3 else i for i, n in enumerate(lengths) for _ in range(n)]
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    ranks = [pick.choice([1, 5, 8, 13, rank // 2, rank]) if mixed else rank for _ in range(slots)]
    shown_a, shown_b = [t.clone() for t in a], [t.clone() for t in b]  # what the oracle sees: zeros beyond a slot's rank
    for s, r in enumerate(ranks):
        for t, z in zip(a, shown_a):
            t[s, r:], z[s, r:] = float("nan"), 0
        for t, z in zip(b, shown_b):
            t[s, :, r:], z[s, :, r:] = float("nan"), 0
    dev = [t.cuda() for t in a], [t.cuda() for t in b]
    eff = torch.tensor(ranks, dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices.cuda(), slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, dtype), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    runs = []
    try:
        monkeypatch.setenv("MLORA_SLAB", "2")
        monkeypatch.setenv("MLORA_SGMV_KSPLIT", str(parts))
        _hip.reload_knobs()
        for _ in range(2):
            out = y.cuda()
            _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, _hip.FORM_SGMV, scratch, effective_rank=eff)
            runs.append(out.cpu())
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(runs[0], runs[1])
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"slab {CASES[case]}")
