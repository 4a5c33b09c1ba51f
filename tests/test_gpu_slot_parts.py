"""The slot-major form with K = 8192 shared out between eight workgroups of a tile, at the sizes where it can go
wrong: one token, full and further tiles of a slot, parts of 64 to 512 output columns, a last part that is short,
every rank, adapters below the buffers' rank; the same bits whether partners' words are accepted or not."""

import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
CASES = [  # tokens, slots, rank, columns, element type, adapters of lower rank
    (1, 1, 8, 512, B16, False),
    (16, 8, 16, 2048, F16, False),
    (40, 3, 24, 1016, B16, False),
    (70, 9, 32, 2248, B16, True),
    (33, 2, 64, 4096, F16, False),
    (20, 5, 48, 2048, B16, True),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_eight_parts_of_k_against_fp64(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    tokens, slots, rank, n, dtype, mixed = CASES[case]
    k = 8192
    print(f"eight parts {CASES[case]}", flush=True)
    g = torch.Generator().manual_seed(case)
    indices = torch.randint(-1, slots, (tokens,), generator=g, dtype=torch.int32)
    indices[0] = slots - 1
    indices[tokens // 2 :] = 0  # a slot of several tiles
    a, b = (torch.randn(slots, rank, k, generator=g) * 0.02).to(dtype), (torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype)
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, n, generator=g).to(dtype)
    ranks = [(5, rank, 8, rank // 2)[s % 4] if mixed else rank for s in range(slots)]
    for s, r in enumerate(ranks):
        a[s, r:], b[s, :, r:] = 0, 0
    eff = torch.tensor(ranks, dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices.cuda(), slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, 1, rank, dtype), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    runs = []
    try:
        for ticks in ("20000", "20000", "-1"):
            monkeypatch.setenv("MLORA_SLOT_SPIN_TICKS", ticks)
            _hip.reload_knobs()
            out = y.cuda()
            _hip.add_lora(out, x.cuda(), [a.cuda()], [b.cuda()], [0], indices.cuda(), plan.workspace, 0.75, _hip.FORM_SLOT, scratch, effective_rank=eff)
            runs.append(out.cpu())
            if ticks != "-1":
                assert scratch.view(torch.int32)[_hip.WORKSPACE_TIMEOUTS_WORD].item() == 0, "a wait ran out"
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
    assert torch.equal(runs[0][indices < 0], y[indices < 0])
    exact, mag = _exact(types.SimpleNamespace(a=[a], b=[b], widths=[n]), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"eight parts {CASES[case]}")
