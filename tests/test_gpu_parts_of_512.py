"""K = 2048 and 4096 shared out between four and eight workgroups of four wavefronts, against fp64: one slice and three, one and two
column spans per wavefront, a last part with fewer columns, buffers of a rank between the instances', further tiles of a slot; the same bits
with the partners' words accepted and never accepted; the workspace's eight states one generation on per launch, and a state
that fits no launch neither believed nor touched."""

import types

import pytest
import torch

from test_gpu_parity import _check, _exact

B16, F16 = torch.bfloat16, torch.float16
CASES = [  # k, tokens, slots, rank, n, dtype, mixed ranks
    (2048, 1, 8, 64, 2048, B16, False),
    (2048, 70, 24, 32, 1024, F16, True),
    (2048, 90, 5, 24, 1000, B16, False),
    (2048, 200, 48, 8, 512, F16, False),
    (2048, 33, 9, 64, 2048, F16, True),
    (2048, 41, 16, 64, (2048, 512, 512), F16, True),
    (2048, 3, 5, 64, (1000, 392, 512), B16, False),
    (4096, 40, 16, 16, 1024, B16, False),
    (4096, 33, 8, 64, 2048, F16, True),
    (4096, 20, 5, 32, 4096, B16, False),
    (4096, 2, 24, 48, 1000, B16, True),
    (2048, 35, 12, 48, 1000, F16, True),
]
_STATES = [64] + [(256 + 8192 + 256 * x) // 4 for x in range(1, 8)]  # first words of the states


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_fp64(case, monkeypatch):
    from nanovllm_voxcpm_amd import _hip
    from nanovllm_voxcpm_amd.lora_ops.segment_meta import build_segment_plan

    k, tokens, slots, rank, n, dtype, mixed = CASES[case]
    print(f"parts of 512 {CASES[case]}", flush=True)
    g = torch.Generator().manual_seed(case)
    indices = torch.randint(-1, slots, (tokens,), generator=g, dtype=torch.int32)
    indices[0] = slots - 1
    indices[tokens // 2 + 1 :] = 0  # a slot of several tiles
    widths = list(n) if isinstance(n, tuple) else [n]
    a, b = [(torch.randn(slots, rank, k, generator=g) * 0.02).to(dtype) for _ in widths], [(torch.randn(slots, w, rank, generator=g) * 0.1).to(dtype) for w in widths]
    x, y = torch.randn(tokens, k, generator=g).to(dtype), torch.randn(tokens, sum(widths), generator=g).to(dtype)
    ranks = [(5, rank, 8, rank // 2)[s % 4] if mixed else rank for s in range(slots)]
    for s, r in enumerate(ranks):
        for wa, wb in zip(a, b):
            wa[s, r:], wb[s, :, r:] = 0, 0
    eff = torch.tensor(ranks, dtype=torch.int32, device="cuda") if mixed else None
    plan = build_segment_plan(indices.cuda(), slots)
    scratch = torch.empty(_hip.add_workspace_bytes(tokens, len(widths), rank, dtype), dtype=torch.uint8, device="cuda")
    _hip.workspace_init(scratch)
    head = scratch[: _hip.WORKSPACE_HEAD_BYTES].view(torch.int32)

    def state(at):
        return [v % (1 << 32) for v in head[at : at + 3].tolist()]

    runs = []

    def run(ticks):
        monkeypatch.setenv("MLORA_SLOT_SPIN_TICKS", ticks)
        _hip.reload_knobs()
        out = y.cuda()
        _hip.add_lora(out, x.cuda(), [t.cuda() for t in a], [t.cuda() for t in b], [sum(widths[:i]) for i in range(len(widths))], indices.cuda(),
                      plan.workspace, 0.75, _hip.FORM_SLOT, scratch, effective_rank=eff)
        runs.append(out.cpu())
        if ticks != "-1":
            assert head[_hip.WORKSPACE_TIMEOUTS_WORD].item() == 0, "a wait ran out"
        return len(runs)

    try:
        for ticks in ("20000", "20000", "-1", "20000"):
            count = run(ticks)
            assert all(state(at) == [count, 0, count ^ 0x9E3779B9] for at in _STATES)
        for wrong in ([9, 0, count ^ 0x9E3779B9], [count, 1 << 20, count ^ 0x9E3779B9]):
            head[_STATES[0] : _STATES[0] + 3] = torch.tensor([(v + (1 << 31)) % (1 << 32) - (1 << 31) for v in wrong], dtype=torch.int32, device="cuda")
            run("20000")
            assert state(_STATES[0]) == wrong
    finally:
        monkeypatch.undo()
        _hip.reload_knobs()
    assert all(torch.equal(runs[0], other) for other in runs[1:])
    assert torch.equal(runs[0][indices < 0], y[indices < 0])
    exact, mag = _exact(types.SimpleNamespace(a=a, b=b, widths=widths), x, y, indices, 0.75)
    _check(runs[0], y, exact, mag, indices, f"parts of 512 {CASES[case]}")
