"""Tiles whose wavefronts request one, two or four token rows per lane group (csrc/slot.hip, csrc/decode.hip): every count of
tokens around the lines, both grids, every rank, one span per wavefront, two and more, every staged K, adapters below the buffers' rank
with NaN beyond it.  In the grid over tiles the texts for short tiles are launched by force, and leave the bits of the one text."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
COUNTS = [1, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 0, 21, 24, 25, 32]

# rank, K, widths, element type, adapters of lower rank, columns per range (0: the library's)
CASES = [
    (8, 1024, [72], B16, False, 0),
    (16, 1024, [512, 64], F16, False, 0),
    (32, 1024, [264], B16, True, 0),
    (64, 1024, [1024, 256, 256], B16, True, 0),
    (16, 2048, [520], B16, False, 0),
    (16, 4096, [512], F16, True, 0),
    (48, 1024, [1000], B16, True, 0),
    (8, 2048, [1000], B16, False, 1024),
    (8, 3072, [520], F16, True, 512),
    (8, 4096, [72], B16, False, 512),
    (16, 1024, [2104], B16, True, 2048),
    (16, 2048, [1032], F16, True, 1024),
    (16, 3072, [1032], B16, False, 1024),
    (16, 4096, [1032], B16, True, 1024),
    (24, 1024, [1032], F16, True, 1024),
    (32, 1024, [2104], B16, False, 2048),
    (32, 2048, [520], F16, True, 512),
    (32, 2048, [1032], B16, False, 1024),
    (64, 1024, [1032], F16, True, 1024),
    (56, 1024, [264], F16, False, 0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_every_count_of_tokens(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    rank, k, widths, dtype, mixed, columns = CASES[case]
    print(f"short tiles {CASES[case]}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    slots = len(COUNTS)
    ids = [i for i, n in enumerate(COUNTS) for _ in range(n)] + [-1] * 3
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
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)

    def run(form):
        out = y.cuda()
        _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, form, scratch, effective_rank=eff)
        return out.cpu()

    runs = {}
    try:
        monkeypatch.setenv("MLORA_DECODE_NT", str(columns))
        for name, texts in (("short", 1), ("short again", 1), ("one text", 0), ("the library's", -1)):
            monkeypatch.setenv("MLORA_DECODE_SHORT", str(texts))
            _hip.reload_knobs()
            runs[name] = run(_hip.FORM_MFMA)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    for name, out in runs.items():
        assert torch.equal(out, runs["one text"]), name
    if k == 1024 and max(widths) <= 1032 and not (len(widths) == 3 and rank == 48):
        runs["slots"], again = run(_hip.FORM_SLOT), run(_hip.FORM_SLOT)
        assert torch.equal(runs["slots"], again)
    for name, out in runs.items():
        assert torch.equal(out[indices < 0], y[indices < 0])
        _check(out, y, exact, mag, indices, f"short tiles {CASES[case]}, {name}")
