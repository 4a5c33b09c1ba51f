"""The shrink through LDS (csrc/slab.hip) at rank 64, one or two slices, at the sizes where it can go wrong: K of
fewer 128-byte pieces per wavefront than the ring has stages, tiles of every number of 16-token blocks, uneven K
parts, adapters below the buffers' rank with NaN beyond it; and which shrink, in how many K parts, the automatic choice takes on both
sides of its lines."""

import random
import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16

# segment lengths, K, widths, element type, adapters of lower rank, every fourth segment without adapter, K parts of this shrink (None: forced, 0: the
# automatic choice is the other shrink)
CASES = [
    ([64], 128, [8], B16, False, False, None),
    ([16, 17, 1, 15], 128, [520, 64], F16, False, False, None),
    ([32, 33, 48, 49, 3], 384, [264], B16, True, True, None),
    ([130, 20, 64, 31, 5], 2560, [512], F16, True, True, None),
    ([257, 16, 90], 4096, [72, 200], B16, True, False, None),
    ([2100, 2400], 2560, [2560], B16, False, False, 2),  # parts of 1280, where the other shrink does not cut K
    ([1500, 1700, 1300], 4096, [1024], F16, True, False, 0),  # three parts, where the other shrink has four
    ([1600, 1701, 1599], 3072, [1024], B16, False, False, 3),  # up to ten workgroups an XCD and part
    ([800] * 5 + [1000], 3072, [1024], B16, False, False, 0),  # up to eleven: three parts would be a second round, two are no more than the other's
    ([800] * 5 + [1000], 2560, [1024], F16, True, False, 2),
    ([1000, 2200], 2560, [2560, 2560], B16, False, False, 2),
    ([1000, 2200], 2048, [2048, 2048], B16, False, False, 0),
    ([250] * 14, 2560, [2560], B16, False, False, 0),  # short segments
    ([1000, 900, 900, 1296], 2048, [2048], B16, False, True, 0),  # fewer tiles than tokens / 64: a third of the tokens has none
    ([1300] * 4, 4096, [1024], F16, False, True, 0),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_rank_64_through_lds_against_fp64(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    lengths, k, widths, dtype, mixed, holes, parts = CASES[case]
    print(f"slab, rank 64 {case} {k} {widths}", flush=True)
    pick, g = random.Random(case), torch.Generator().manual_seed(case)
    slots, rank = len(lengths), 64
    ids = [-1 if holes and i % 4 == 3 else i for i, n in enumerate(lengths) for _ in range(n)]
    pick.shuffle(ids)
    indices, tokens = torch.tensor(ids, dtype=torch.int32), len(ids)
    a = [(torch.randn(slots, rank, k, generator=g) * 0.05).to(dtype) for _ in widths]
    b = [(torch.randn(slots, n, rank, generator=g) * 0.1).to(dtype) for n in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    ranks = [pick.choice([1, 8, 13, 32, 64]) if mixed else rank for _ in range(slots)]
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

    def run(form, slab=None, ksplit=None):
        for name, value in (("MLORA_SLAB", slab), ("MLORA_SGMV_KSPLIT", ksplit)):
            monkeypatch.delenv(name, raising=False)
            if value is not None:
                monkeypatch.setenv(name, str(value))
        _hip.reload_knobs()
        out = y.cuda()
        _hip.add_lora(out, x.cuda(), *dev, cols, indices.cuda(), plan.workspace, 0.75, form, scratch, effective_rank=eff)
        return out.cpu()

    try:
        if parts is None:
            runs = [run(_hip.FORM_SGMV, 2) for _ in range(2)]
        else:
            runs = [run(_hip.FORM_AUTO) for _ in range(2)]
            # which shrink that was, by the order in which it adds K up
            others = {n: run(_hip.FORM_AUTO, 2, n) for n in (2, 3, 4)} | {0: run(_hip.FORM_AUTO, 0)}  # (one part may be two of the other's)
            assert [n for n in sorted(others) if torch.equal(runs[0], others[n])] == [parts]
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert torch.equal(runs[0], runs[1])
    exact, mag = _exact(types.SimpleNamespace(a=shown_a, b=shown_b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"slab, rank 64 {case}")
