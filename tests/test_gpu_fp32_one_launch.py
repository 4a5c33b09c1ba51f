"""fp32 over 16-token tiles in one launch (csrc/pair.hip) at the sizes where it can go wrong: one token, full and barely
started tiles, K of fewer 128-byte chunks than wavefronts and of no multiple of them, column counts that end inside a span and
a range, adapters below the buffers' rank with NaN beyond it; and what AUTO takes on both sides of its line."""

import random

import pytest
import torch

from oracle import lora_apply as oracle

# tokens, slots, rank, K, widths, columns per range, adapters of lower rank, segments instead of single tokens
CASES = [
    (1, 1, 8, 32, [8], 256, False, False),
    (16, 1, 16, 1024, [1032], 512, True, True),
    (17, 2, 16, 96, [520], 64, False, True),
    (64, 4, 16, 1024, [1024, 256, 256], 256, False, False),
    (77, 3, 32, 544, [1000, 64], 256, True, True),
    (300, 33, 32, 1024, [264], 128, True, False),
    (50, 7, 8, 2048, [72, 136], 512, True, False),
    (40, 2, 16, 4096, [1024], 256, True, False),
]


def _batch(case, seed):
    tokens, slots, rank, k, widths, _, mixed, segments = case
    pick, g = random.Random(seed), torch.Generator().manual_seed(seed)
    ids = []
    while len(ids) < tokens:
        ids += [pick.randrange(-1, slots)] * (pick.randrange(1, 70) if segments else 1)
    ids[0] = slots - 1
    indices = torch.tensor(ids[:tokens], dtype=torch.int32)
    a = [torch.randn(slots, rank, k, generator=g) * 0.05 for _ in widths]
    b = [torch.randn(slots, n, rank, generator=g) * 0.1 for n in widths]
    x, y = torch.randn(tokens, k, generator=g), torch.randn(tokens, sum(widths), generator=g)
    ranks = [pick.choice([1, 5, 8, 13, rank // 2, rank]) if mixed else rank for _ in range(slots)]
    shown_a, shown_b = [t.clone() for t in a], [t.clone() for t in b]  # what the oracle sees: zeros beyond a slot's rank
    for s, r in enumerate(ranks):
        for t, z in zip(a, shown_a):
            t[s, r:], z[s, r:] = float("nan"), 0
        for t, z in zip(b, shown_b):
            t[s, :, r:], z[s, :, r:] = float("nan"), 0
    want = torch.cat(oracle.fused_add_lora(list(y.split(widths, dim=-1)), x, shown_a, shown_b, indices=indices, scaling=0.75,
                                           accumulate=torch.float64), dim=-1)
    return indices, a, b, x, y, torch.tensor(ranks, dtype=torch.int32) if mixed else None, want


def _apply(case, batch, form):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    tokens, slots, rank, _, widths, *_ = case
    indices, a, b, x, y, ranks, _ = batch
    plan = build_segment_plan(indices.cuda(), slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, torch.float32) + (8 << 20), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    cols = [sum(widths[:i]) for i in range(len(widths))]
    out = y.cuda()
    _hip.add_lora(out, x.cuda(), [t.cuda() for t in a], [t.cuda() for t in b], cols, indices.cuda(), plan.workspace, 0.75, form, scratch,
                  effective_rank=None if ranks is None else ranks.cuda())
    return out.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_one_launch_against_fp64(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip

    print(f"fp32 one launch {CASES[case]}", flush=True)
    batch = _batch(CASES[case], case)
    try:
        monkeypatch.setenv("MLORA_SOLO", "2")
        monkeypatch.setenv("MLORA_SOLO_COLS", str(CASES[case][5]))
        _hip.reload_knobs()
        runs = [_apply(CASES[case], batch, _hip.FORM_AUTO) for _ in range(2)]
        monkeypatch.setenv("MLORA_SOLO", "0")
        _hip.reload_knobs()
        pair = _apply(CASES[case], batch, _hip.FORM_AUTO)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    indices, y, want = batch[0], batch[4], batch[6]
    assert torch.equal(*runs)
    assert torch.equal(runs[0][indices < 0], y[indices < 0])
    assert torch.allclose(runs[0], want, rtol=1e-5, atol=2e-5)
    # its chains are shorter than the pair's or as short: no further from the exact sum than a few of its own ulps
    error, other = (runs[0].double() - want.double()).norm(), (pair.double() - want.double()).norm()
    assert error <= 1.1 * other + 1e-7 * want.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("tokens, slots, rank, k, widths, one_launch", [
    (64, 4, 16, 1024, [1024, 256, 256], True),
    (64, 4, 16, 1024, [4096, 4096], True),
    (64, 32, 16, 1024, [4096, 4096], False),  # 16 ranges of 512 columns x 4 tiles of an XCD
    (64, 4, 16, 4096, [1024], False),
    (64, 4, 32, 2048, [1024], False),
])
def test_auto_takes_one_launch_where_it_pays(tokens, slots, rank, k, widths, one_launch, monkeypatch):
    from nanovllm_voxcpm_amd import _hip

    case = (tokens, slots, rank, k, widths, 0, False, False)
    batch = _batch(case, 5)
    try:
        chosen = _apply(case, batch, _hip.FORM_AUTO)
        monkeypatch.setenv("MLORA_SOLO", "0")
        _hip.reload_knobs()
        pair = _apply(case, batch, _hip.FORM_AUTO)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(chosen, pair) != one_launch  # (the forms add K up in different orders)
    assert torch.allclose(chosen, batch[6], rtol=1e-5, atol=2e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("rank", [24, 40, 48, 56])
@pytest.mark.parametrize("tokens, slots, k, widths", [(1, 3, 32, [4]), (17, 2, 1024, [520, 64]), (150, 40, 2080, [256])])
def test_ranks_between_the_instances_are_two_launches_under_auto(rank, tokens, slots, k, widths, monkeypatch):
    from nanovllm_voxcpm_amd import _hip

    case = (tokens, slots, rank, k, widths, 0, tokens > 1, True)
    batch = _batch(case, rank)
    out = _apply(case, batch, _hip.FORM_AUTO)
    assert torch.equal(out[batch[0] < 0], batch[4][batch[0] < 0])
    assert torch.allclose(out, batch[6], rtol=1e-5, atol=2e-5)
    try:
        monkeypatch.setenv("MLORA_NO_PAIR", "1")
        _hip.reload_knobs()
        one_per_token = _apply(case, batch, _hip.FORM_AUTO)
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.allclose(one_per_token, batch[6], rtol=1e-5, atol=2e-5)
    # (the forms add K up in different orders, which one token of 32 columns need not show)
    assert tokens == 1 or not torch.equal(out, one_per_token)
